"""The sampler's work as a serving engine has it do: what is measured when its speed is.

Each case is one pass through the public entry points of the ``hip`` backend on inputs made from a
seed: the per-token call, batched steps over bf16 and fp32 logits with and without penalties, the
probability of drafted ids, speculative verification, log-probabilities, the filtered
distribution and the LM head with its tile statistics. ``exact`` recomputes the real-valued outputs in
64 bits with plain torch.
"""

from __future__ import annotations

import math

import torch

from vinfer_amd.registry import BackendContext
from vinfer_amd.sampler import SAMPLER
from vinfer_amd.sampling import PackedParams, SamplingParams

DEV = torch.device("cuda", 0)
DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}
PENALTIES = (1.05, 0.5, 0.2)  # repetition, presence, frequency
LOGPROB_TOP = 20  # entries per row: the most an API request may ask for


def listed() -> list[dict]:
    return [
        # One sequence decoded on its own, one call per token: the engine's own loop, with the
        # filters a model card recommends. Launches and latency are all there is.
        _token("token_topk", top_k=20, top_p=0.8, temperature=0.7),
        # The same loop with nucleus sampling alone: the kept set depends on the whole row.
        _token("token_topp", top_p=0.95, temperature=0.8),
        # A lightly loaded server: a few sequences with nucleus sampling, inputs new on every step.
        _batch("few_topp", 8, 151936, rows="normal", std=3.0, params="topp"),
        # A vocabulary that is no multiple of anything, so that most rows start off alignment;
        # ordinary sampling with short histories penalised.
        _batch("odd_vocab", 24, 50257, rows="normal", std=2.5, params="topk", history=600),
        # Continuous batching: requests of every kind in one step (greedy, top-k, nucleus),
        # penalised by 2048 tokens of context each; the decode loop keeps the step prepared.
        _batch("mixed_requests", 64, 151936, rows="normal", std=3.0, params="mixed", history=2048, prepared=True),
        # A full decode batch with long contexts: half the rows certain of a token, half flat.
        _batch("full_batch", 256, 151936, rows="peaked_flat", params="minp_topp", history=4096, prepared=True),
        # The largest batch, logits kept in fp32, contexts up to 32768 tokens.
        _batch("largest_fp32", 1024, 151936, dtype="fp32", rows="normal", std=2.0, params="topk", history=32768,
               ragged_history=True, prepared=True),
        # Scoring drafted tokens: the sampled id and the draft's final probability, a large vocabulary.
        _batch("draft_scores", 192, 262144, rows="normal", std=2.5, params="topp", draft=True),
        # Speculative decoding's verification of one drafted token per sequence.
        {"name": "verify", "kind": "verify", "batch": 192, "num_draft": 1, "vocab": 262144, "std": 2.5},
        # An API step with log-probabilities: the sampled token's and the top 20 of each row.
        {"name": "logprobs", "kind": "logprobs", "batch": 256, "vocab": 151936, "dtype": "bf16", "rows": "peaked_flat",
         "std": 1.0},
        # The distribution itself (what a caller inspects, or mixes with another model's).
        {"name": "probs", "kind": "probs", "batch": 32, "vocab": 151936, "dtype": "bf16", "rows": "normal", "std": 3.0,
         "params": "topp"},
        # The LM head of a decode batch: logits and the tile statistics that the draw and the
        # log-probabilities start from.
        {"name": "lm_head", "kind": "lm_head", "batch": 64, "dim": 4096, "vocab": 151936},
    ]


def _token(name, **params) -> dict:
    return {"name": name, "kind": "token", "vocab": 151936, "dtype": "bf16", "std": 3.0, **params}


def _batch(name, batch, vocab, *, dtype="bf16", rows, std=1.0, params, history=0, ragged_history=False, draft=False,
           prepared=False) -> dict:
    return {"name": name, "kind": "batch", "batch": batch, "vocab": vocab, "dtype": dtype, "rows": rows, "std": std,
            "params": params, "history": history, "ragged_history": ragged_history, "draft": draft, "prepared": prepared}


def draw(rng) -> dict:
    def between(lo, hi):  # over the logarithm
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    vocab = between(8000, 262144)
    if rng.random() < 0.6:  # most vocabularies are padded to a multiple of 64
        vocab = min(262144, (vocab + 63) // 64 * 64)
    kind = rng.choices(["token", "batch", "verify", "logprobs", "probs", "lm_head"], [3, 12, 2, 3, 2, 2])[0]
    std = round(rng.uniform(1.0, 4.0), 2)
    if kind == "token":
        c = {"kind": kind, "vocab": vocab, "dtype": rng.choice(["bf16", "bf16", "fp32"]), "std": std,
             "temperature": round(rng.uniform(0.3, 1.3), 2)}
        return {**c, **rng.choice([{"top_k": rng.randint(1, 100), "top_p": 0.9}, {"top_p": round(rng.uniform(0.8, 0.99), 3)},
                                   {"temperature": 0.0}])}
    if kind == "batch":
        dtype = rng.choice(["bf16", "bf16", "bf16", "fp32"])
        params = rng.choice(["greedy", "topk", "topp", "minp_topp", "mixed"])
        if dtype == "fp32" and params != "topk":  # (fp32 rows whose kept set no top-k bounds take many passes)
            params = rng.choice(["greedy", "topk"])
        most = min(1024, int((160e6 if dtype == "bf16" else 320e6) / (vocab * (2 if dtype == "bf16" else 4))))
        history = rng.choice([0, 0, between(16, 8000)])
        return {k: v for k, v in _batch(
            "", between(1, most), vocab, dtype=dtype, rows=rng.choice(["normal", "normal", "peaked_flat"]), std=std,
            params=params, history=history, ragged_history=rng.random() < 0.5, draft=rng.random() < 0.25,
            prepared=rng.random() < 0.5).items() if k != "name"}
    if kind == "verify":
        num_draft = rng.randint(1, 4)
        return {"kind": kind, "batch": between(1, max(2, int(150e6 / (vocab * 2 * (2 * num_draft + 1))))),
                "num_draft": num_draft, "vocab": vocab, "std": std}
    if kind == "logprobs":
        return {"kind": kind, "batch": between(1, max(2, min(512, int(100e6 / (vocab * 2))))), "vocab": vocab,
                "dtype": rng.choice(["bf16", "bf16", "bf16", "fp32"]), "rows": rng.choice(["normal", "peaked_flat"]),
                "std": std}
    if kind == "probs":
        return {"kind": kind, "batch": between(1, max(2, min(128, int(20e6 / (vocab * 2))))), "vocab": vocab,
                "dtype": "bf16", "rows": rng.choice(["normal", "peaked_flat"]), "std": std,
                "params": rng.choice(["topk", "topp", "minp_topp"])}
    dim = rng.choice([512, 1024, 2048, 3072, 4096])
    return {"kind": kind, "batch": between(1, 64), "dim": dim, "vocab": min(vocab, 151936)}


# ---- inputs ---------------------------------------------------------------------------------------
def _rng(seed: int) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _backend(dtype: torch.dtype):
    return SAMPLER.resolve("hip", BackendContext(DEV, dtype))


def _logits(g, batch, vocab, dtype, rows, std):
    x = torch.randn(batch, vocab, generator=g, device=DEV) * (std if rows == "normal" else 1.0)
    if rows == "peaked_flat":  # even rows certain of one token, odd rows nearly uniform
        x[1::2] *= 0.1
        even = torch.arange(0, batch, 2, device=DEV)
        x[even, torch.randint(0, vocab, even.shape, generator=g, device=DEV)] += 15.0
    return x.to(DTYPES[dtype])


def _uniforms(g, *shape):
    return torch.rand(*shape, generator=g, device=DEV)


def _params(g, batch, kind, penalised) -> PackedParams:
    def f32(v):
        return v.float() if isinstance(v, torch.Tensor) else torch.full((batch,), float(v), device=DEV)

    temperature, top_k, top_p, min_p = 0.8, torch.zeros(batch, device=DEV), 1.0, 0.0
    if kind == "greedy":
        temperature = 0.0
    elif kind == "topk":
        top_k, top_p = torch.full((batch,), 50.0, device=DEV), 0.9
    elif kind == "topp":
        temperature, top_p = 0.5 + 0.7 * _uniforms(g, batch), 0.95
    elif kind == "minp_topp":
        temperature, top_p, min_p = 1.0, 0.95, 0.05
    elif kind == "mixed":
        greedy = _uniforms(g, batch) < 0.25
        temperature = torch.where(greedy, 0.0, 0.3 + 1.2 * _uniforms(g, batch))
        top_k = torch.tensor([0.0, 20.0, 50.0, 1000.0], device=DEV)[torch.randint(0, 4, (batch,), generator=g, device=DEV)]
        top_p = 0.5 + 0.5 * _uniforms(g, batch)
    else:
        raise ValueError(f"unknown parameters {kind!r}")
    rep, pres, freq = PENALTIES if penalised else (1.0, 0.0, 0.0)
    return PackedParams(temperature=f32(temperature), top_k=top_k.to(torch.int32), top_p=f32(top_p), min_p=f32(min_p),
                        repetition_penalty=f32(rep), presence_penalty=f32(pres), frequency_penalty=f32(freq))


def _histories(g, batch, vocab, length, ragged):
    """Token ids by Zipf's law (ranks mapped to ids by a permutation), as text has them, in CSR form."""
    lengths = (torch.randint(1, length + 1, (batch,), generator=g, device=DEV) if ragged
               else torch.full((batch,), length, dtype=torch.int64, device=DEV))
    offsets = torch.zeros(batch + 1, dtype=torch.int64, device=DEV)
    torch.cumsum(lengths, 0, out=offsets[1:])
    cdf = torch.cumsum(torch.arange(1, vocab + 1, device=DEV, dtype=torch.float64) ** -1.1, 0)
    total = int(offsets[-1])
    u = torch.rand(total, generator=g, device=DEV, dtype=torch.float64) * cdf[-1]
    ranks = torch.searchsorted(cdf, u).clamp_(max=vocab - 1)
    perm = torch.randperm(vocab, generator=g, device=DEV)
    return perm[ranks].to(torch.int32), offsets.to(torch.int32)


def _inputs(case, seed) -> dict:
    """Every input of the case, the same for ``prepare`` and ``exact``."""
    g, kind = _rng(seed), case["kind"]
    if kind == "lm_head":
        hidden = torch.randn(case["batch"], case["dim"], generator=g, device=DEV)
        weight = torch.randn(case["vocab"], case["dim"], generator=g, device=DEV, dtype=torch.bfloat16)
        weight *= 3.0 / math.sqrt(case["dim"])
        return {"hidden": hidden.to(torch.bfloat16), "weight": weight}
    if kind == "token":
        return {"logits": _logits(g, 1, case["vocab"], case["dtype"], "normal", case["std"])[0]}
    batch, vocab = case["batch"], case["vocab"]
    if kind == "verify":
        k = case["num_draft"]
        # the draft model's logits: the target's at the same position with noise, so that most
        # drafts are accepted
        target = torch.randn(batch, k + 1, vocab, generator=g, device=DEV) * case["std"]
        draft = target[:, :k] + 0.5 * torch.randn(batch, k, vocab, generator=g, device=DEV)
        return {"target": target.to(torch.bfloat16), "draft": draft.to(torch.bfloat16),
                "params": _params(g, batch, "topp", False), "u_draft": _uniforms(g, batch * k),
                "u_accept": _uniforms(g, batch, k), "u_residual": _uniforms(g, batch, k), "u_bonus": _uniforms(g, batch)}
    x = {"logits": _logits(g, batch, vocab, case["dtype"], case["rows"], case["std"])}
    if kind == "logprobs":
        return {**x, "tokens": torch.randint(0, vocab, (batch,), generator=g, device=DEV).to(torch.int32)}
    history = case.get("history", 0)
    x["params"] = _params(g, batch, case["params"], history > 0)
    if kind == "batch":
        x["uniforms"] = _uniforms(g, batch)
        x["hist_ids"] = x["hist_offsets"] = x["draft_ids"] = None
        if history:
            x["hist_ids"], x["hist_offsets"] = _histories(g, batch, vocab, history, case["ragged_history"])
        if case["draft"]:  # the draft model's best token
            noisy = x["logits"].float()
            noisy += torch.randn(batch, vocab, generator=g, device=DEV)
            x["draft_ids"] = noisy.argmax(dim=1).to(torch.int32)
    return x


def prepare(case, seed):
    kind = case["kind"]
    state = {"kind": kind, "backend": _backend(DTYPES[case.get("dtype", "bf16")]), **_inputs(case, seed)}
    s = state["backend"]
    if kind == "token":
        state["params"] = SamplingParams(temperature=case["temperature"], top_k=case.get("top_k", 0),
                                         top_p=case.get("top_p", 1.0), seed=int(seed))
        state["seed"] = int(seed)
    elif kind == "batch" and case["prepared"]:
        state["step"] = s.prepare_batch(*(state[k] for k in ("logits", "params", "uniforms", "hist_ids", "hist_offsets",
                                                             "draft_ids")))
    elif kind == "verify":  # the drafter has drawn its tokens, and kept their rows' states
        rows = state["draft"].reshape(-1, case["vocab"])
        drafts, states = s.sample_states(rows, state["params"].repeat_rows(case["num_draft"]), state["u_draft"])
        state["drafts"], state["states"] = drafts.view(case["batch"], -1), states
    return state


def run(state):
    s, kind = state["backend"], state["kind"]
    if kind == "token":
        return s.sample(state["logits"], state["params"], state["seed"], 17)
    if kind == "batch":
        step = state.get("step")
        if step is not None:
            step.launch()
            return step.ids, step.draft_prob
        return s.sample_batch(state["logits"], state["params"], state["uniforms"], state["hist_ids"],
                              state["hist_offsets"], state["draft_ids"])
    if kind == "verify":
        return s.verify(state["target"], state["draft"], state["drafts"], state["params"], state["u_accept"],
                        state["u_residual"], state["u_bonus"], draft_states=state["states"])
    if kind == "logprobs":
        return s.logprobs(state["logits"], state["tokens"], LOGPROB_TOP)
    if kind == "probs":
        return s.probs(state["logits"], state["params"])
    return s.lm_head(state["hidden"], state["weight"])


def work(case):
    kind, vocab = case["kind"], case["vocab"]
    size = 4 if case.get("dtype") == "fp32" else 2
    if kind == "token":
        return {"bytes": vocab * size + 36, "flops": 0}
    batch = case["batch"]
    if kind == "lm_head":
        dim = case["dim"]
        tiles = (vocab + 127) // 128
        return {"bytes": 2 * vocab * dim + 2 * batch * dim + 2 * batch * vocab + 8 * batch * tiles,
                "flops": 2 * batch * dim * vocab}
    if kind == "verify":
        k = case["num_draft"]
        return {"bytes": size * batch * (2 * k + 1) * vocab + batch * (64 * k + 40), "flops": 0}
    if kind == "logprobs":
        return {"bytes": size * batch * vocab + batch * (8 + 8 * LOGPROB_TOP), "flops": 0}
    if kind == "probs":
        return {"bytes": batch * vocab * (size + 4) + 28 * batch, "flops": 0}
    history = case["history"] * (0.5 if case["ragged_history"] else 1.0)
    return {"bytes": int(batch * (size * vocab + 4 * history + 40)), "flops": 0}


def tolerance(case):
    kind = case["kind"]
    if kind == "lm_head":
        # bf16 logits, rounded from fp32 sums in any order: a few in a thousand land on the other
        # side of a rounding boundary, one unit in the last place (2**-8 of the value) apart
        return {"rel": 1e-3, "max": 0.016}
    if kind == "logprobs":  # fp32 exponentials summed in any order; the ids exactly
        return {"rel": 2e-6, "max": 1e-5}
    if kind == "probs" or case.get("draft"):  # fp64 exponentials, rounded to fp32 once
        return {"rel": 1e-6, "max": 1e-5}
    return "exact"  # token ids


# ---- the same in 64 bits ------------------------------------------------------------------------
def _distribution(x, p: PackedParams, hist_ids=None, hist_offsets=None):
    """The fp64 probabilities a row is drawn from, rows ``[B, V]``."""
    batch, vocab = x.shape
    z = x.double()
    if hist_ids is not None:
        counts = torch.zeros(batch * vocab, dtype=torch.float64, device=DEV)
        row = torch.repeat_interleave(torch.arange(batch, device=DEV), hist_offsets.long().diff())
        counts.index_add_(0, row * vocab + hist_ids.long(), torch.ones(row.shape[0], dtype=torch.float64, device=DEV))
        counts = counts.view(batch, vocab)
        rep, pres, freq = (v.double()[:, None] for v in (p.repetition_penalty, p.presence_penalty, p.frequency_penalty))
        z = torch.where(counts > 0, torch.where(z > 0, z / rep, z * rep) - freq * counts - pres, z)
    greedy = p.temperature <= 0
    first = z.argmax(dim=1)
    z = z / torch.where(greedy, 1.0, p.temperature.double())[:, None]
    order = z.argsort(dim=1, descending=True, stable=True)
    zs = z.gather(1, order)
    k = torch.where((p.top_k > 0) & (p.top_k < vocab), p.top_k, vocab).long()
    w = torch.where(zs >= zs.gather(1, k[:, None] - 1), (zs - zs[:, :1]).exp(), 0.0)
    w = torch.where(w >= p.min_p.double()[:, None], w, 0.0)
    before = w.cumsum(1) - w
    w = torch.where((before < p.top_p.double()[:, None] * w.sum(1, keepdim=True)) | (p.top_p >= 1)[:, None], w, 0.0)
    out = torch.zeros_like(z).scatter_(1, order, w / w.sum(1, keepdim=True))
    out[greedy] = torch.nn.functional.one_hot(first[greedy], vocab).double()
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind in ("token", "verify"):
        return None  # token ids alone
    x = _inputs(case, seed)
    if kind == "lm_head":
        hidden = x["hidden"].double().t().contiguous()
        logits = torch.cat([(w.double() @ hidden).t() for w in x["weight"].split(16384)], dim=1)
        pad = -case["vocab"] % 128
        tiles = torch.nn.functional.pad(logits, (0, pad), value=-math.inf).view(case["batch"], -1, 128)
        top = tiles.amax(dim=2)
        return logits, top, (tiles - top[:, :, None]).exp().sum(dim=2)
    if kind == "logprobs":
        lp = torch.log_softmax(x["logits"].double(), dim=1)
        return lp.gather(1, x["tokens"].long()[:, None])[:, 0], None, lp.topk(LOGPROB_TOP, dim=1).values
    if kind == "probs":
        return _distribution(x["logits"], x["params"])
    if not case["draft"]:
        return None
    out = []
    for rows in torch.arange(case["batch"], device=DEV).split(32):
        hist = ()
        if x["hist_ids"] is not None:
            o = x["hist_offsets"][rows[0]:rows[-1] + 2]
            hist = x["hist_ids"][o[0]:o[-1]], o - o[0]
        p = _distribution(x["logits"][rows], x["params"].select(rows), *hist)
        out.append(p.gather(1, x["draft_ids"][rows].long()[:, None])[:, 0])
    return None, torch.cat(out)
