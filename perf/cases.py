"""The sampling work that this package's speed is measured on.

A case is one call through a public entry point on device-resident logits ``[batch, vocab]``:

* ``op="sample"``: ``ops.prepare_sample(...)`` once per set of buffers (a serving loop keeps its
  logits buffer, parameter tensors and outputs), then ``launch()`` per step;
* ``op="forward"``: the vLLM-v1 front end, ``Sampler.forward(logits, metadata)``, greedy;
* ``op="softmax"`` and ``op="topk"``: the standalone operations.

Vocabularies are those of the models the package's workloads are shaped after (32 000, 128 256,
151 936, 262 144) and anything between; batches go from one request to 1024.  Logits are
N(0, spread) plus, per case, a Zipf-like bias over a shuffled vocabulary (``zipf``) or ``spikes``
tokens per row lifted by ``lift``, which is what a confident model's rows look like.

Tokens, survivor counts, ids and ranks are whole numbers and must not change.  The row flags are
left out of the outputs: their upper bits say which internal path served a row and are
diagnostic by the library's own contract.
"""
from __future__ import annotations

import math

import torch

from vllm_webgpu_amd import ops
from vllm_webgpu_amd.v1.sample.metadata import SamplingMetadata
from vllm_webgpu_amd.v1.sample.sampler import Sampler

_DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}

_BASE = {
    "op": "sample", "batch": 1, "vocab": 32000, "dtype": "f32",
    "spread": 3.0, "zipf": 0.0, "spikes": 0, "lift": 0.0,
    "temperature": 1.0, "top_k": 0, "top_p": 1.0, "min_p": 0.0, "mixed": False,
    "history": 0, "bans": 0, "allowed": 0.0, "softcap": 0.0,
    "logprobs": -1, "uniforms": "generated",
}


def _case(name=None, **kw):
    c = dict(_BASE, **kw)
    if name is not None:
        c["name"] = name
    return c


def listed():
    return [
        # one greedy request on a small vocabulary, through the v1 front end: latency and host
        # work of the smallest step
        _case("greedy_one", op="forward", vocab=32000, spread=2.0, spikes=5, lift=8.0, temperature=0.0),
        # one chat request, temperature and top-p only (a chat model's usual defaults)
        _case("chat_one", vocab=128256, spread=2.0, spikes=12, lift=9.0, temperature=0.6, top_p=0.9),
        # a small batch on a small vocabulary: top-k and top-p, the caller's uniforms
        _case("batch64_topk_topp", batch=64, vocab=32000, zipf=1.1, temperature=0.8, top_k=50,
              top_p=0.9, uniforms="given"),
        # the headline workload: a full batch with penalties over a 512-token history
        _case("batch256_penalties", batch=256, vocab=128256, temperature=0.7, top_k=50, top_p=0.9,
              history=512, uniforms="given"),
        # heterogeneous requests on the largest vocabulary, 16-bit logits: greedy, top-k and
        # top-p-only rows, some with min-p
        _case("mixed512_bf16", batch=512, vocab=262144, dtype="bf16", spread=4.0, spikes=10, lift=10.0,
              mixed=True, uniforms="given"),
        # a large decode batch that returns the top 20 logprobs
        _case("batch1024_logprobs", batch=1024, vocab=151936, zipf=1.2, top_p=0.95, logprobs=20,
              uniforms="given"),
        # the sampling defaults (temperature 1, nothing cut), as rollouts run
        _case("plain128_bf16", batch=128, vocab=151936, dtype="bf16", zipf=1.1),
        # a small batch of a soft-capped model, half-precision logits, its top-k/top-p defaults
        _case("softcap16_f16", batch=16, vocab=262144, dtype="f16", spread=5.0, spikes=10, lift=18.0,
              top_k=64, top_p=0.95, softcap=30.0),
        # structured output: every row carries a grammar's allowed-token mask
        _case("masked32_bf16", batch=32, vocab=151936, dtype="bf16", temperature=0.7, top_k=20,
              top_p=0.8, allowed=0.05),
        # top-p requests whose penalties come from id lists, with stop ids banned (min-tokens)
        _case("topp48_idlists", batch=48, vocab=151936, spread=2.0, spikes=40, lift=8.0, temperature=0.8,
              top_p=0.95, history=512, bans=4),
        # probabilities of a batch, with a temperature
        _case("softmax32", op="softmax", batch=32, vocab=128256, spread=2.0, temperature=0.8),
        # the candidates of a small batch (speculative drafts, beams)
        _case("topk16_bf16", op="topk", batch=16, vocab=128256, dtype="bf16", top_k=20),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    vocab = rng.choice([32000, 128256, 151936, 262144, _log_int(rng, 32000, 262144),
                        _log_int(rng, 32000, 262144) | 1])
    dtype = rng.choice(["f32", "bf16", "f16"])
    kind = rng.choice(["greedy", "topk", "topk", "topp", "topp", "plain", "mixed", "softcap", "masked",
                       "idlists", "softmax", "topk_op"])
    most = 48 if kind in ("idlists", "softcap") else 256 if kind in ("softmax", "plain", "mixed") else 1024
    batch = min(_log_int(rng, 1, most), (1 << 27) // vocab)
    kw = {"batch": max(1, batch), "vocab": vocab, "dtype": dtype}
    shape = rng.choice([{"zipf": round(rng.uniform(1.0, 1.3), 3)},
                        {"spread": 2.0, "spikes": rng.randint(5, 40), "lift": round(rng.uniform(6.0, 10.0), 2)}])
    kw.update(shape)
    some_t, some_p = round(rng.uniform(0.4, 1.3), 3), round(rng.uniform(0.7, 0.98), 3)
    some_u = rng.choice(["given", "generated"])
    if kind == "greedy":
        return _case(op="forward", temperature=0.0, **kw)
    if kind == "topk":
        return _case(temperature=some_t, top_k=rng.randint(5, 100), top_p=rng.choice([1.0, some_p]),
                     history=rng.choice([0, 256, 512]), logprobs=rng.choice([-1, -1, 5, 20]),
                     uniforms=some_u, **kw)
    if kind == "topp":
        return _case(temperature=some_t, top_p=some_p, min_p=rng.choice([0.0, 0.0, 0.05]),
                     logprobs=rng.choice([-1, -1, 5, 20]), uniforms=some_u, **kw)
    if kind == "plain":
        return _case(temperature=rng.choice([1.0, some_t]), uniforms=some_u, **kw)
    if kind == "mixed":
        return _case(mixed=True, uniforms=some_u, **kw)
    if kind == "softcap":
        kw.update(spread=5.0, zipf=0.0, spikes=10, lift=18.0)
        return _case(temperature=some_t, top_k=rng.randint(20, 64), top_p=some_p, softcap=30.0, **kw)
    if kind == "masked":
        return _case(temperature=some_t, top_k=rng.randint(5, 50), top_p=some_p,
                     allowed=rng.choice([0.01, 0.05, 0.5]), **kw)
    if kind == "idlists":
        return _case(temperature=some_t, top_p=some_p, history=rng.choice([128, 512, 700]),
                     bans=rng.choice([0, 4]), **kw)
    if kind == "softmax":
        return _case(op="softmax", temperature=some_t, **kw)
    return _case(op="topk", top_k=rng.randint(1, 100), **kw)


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 13)


def _inputs(case, seed):
    """The tensors of one case, by name, from the seed alone (no code of this package)."""
    g = _generator(seed)
    dev, B, V = "cuda", case["batch"], case["vocab"]
    x = torch.randn((B, V), generator=g, device=dev).mul_(case["spread"])
    if case["zipf"]:
        rank = torch.randperm(V, generator=g, device=dev).add_(1).float()
        x -= case["zipf"] * rank.log()
    if case["spikes"]:
        at = torch.randint(V, (B, case["spikes"]), generator=g, device=dev)
        x.scatter_(1, at, x.gather(1, at) + case["lift"])
    t = {"logits": x.to(_DTYPES[case["dtype"]])}
    del x
    full = lambda v, d=torch.float32: torch.full((B,), v, dtype=d, device=dev)  # noqa: E731
    if case["op"] == "softmax":
        t["temperature"] = full(case["temperature"])
    if case["op"] != "sample":
        return t
    rand = lambda: torch.rand(B, generator=g, device=dev)  # noqa: E731
    if case["mixed"]:
        temp = rand() * 1.5
        temp[torch.randperm(B, generator=g, device=dev)[: B // 8]] = 0.0
        ks = torch.tensor([0, 20, 100], dtype=torch.int32, device=dev)
        t["temperature"] = temp
        t["top_k"] = ks[torch.randint(3, (B,), generator=g, device=dev)]
        t["top_p"] = 0.5 + 0.5 * rand()
        t["min_p"] = torch.where(rand() < 0.5, 0.0, 0.05).float()
    else:
        t["temperature"] = full(case["temperature"])
        t["top_k"] = full(case["top_k"], torch.int32) if case["top_k"] else None
        t["top_p"] = full(case["top_p"]) if case["top_p"] < 1.0 else None
        t["min_p"] = full(case["min_p"]) if case["min_p"] else None
    if case["history"]:
        t["output_ids"] = torch.randint(V, (B, case["history"]), generator=g, device=dev, dtype=torch.int32)
        t["repetition_penalty"], t["presence_penalty"], t["frequency_penalty"] = full(1.1), full(0.5), full(0.3)
    if case["bans"]:
        t["adjust_ids"] = torch.randint(V, (B, case["bans"]), generator=g, device=dev, dtype=torch.int32)
        t["adjust_vals"] = torch.full((B, case["bans"]), float("-inf"), device=dev)
    if case["allowed"]:
        keep = torch.rand((B, -(-V // 32), 32), generator=g, device=dev) < case["allowed"]
        weight = torch.bitwise_left_shift(torch.ones(32, dtype=torch.int64, device=dev),
                                          torch.arange(32, device=dev))
        words = (keep.long() * weight).sum(2)
        t["allowed_mask"] = torch.where(words >= 2 ** 31, words - 2 ** 32, words).int()
    if case["softcap"]:
        t["logit_softcap"], t["logit_softcap_f16"] = case["softcap"], case["dtype"] == "f16"
    if case["uniforms"] == "given":
        # multiples of 2^-24 in (0, 1), as the kernel's own are
        t["uniforms"] = torch.rand((B, V), generator=g, device=dev).clamp_(2.0 ** -24, 1.0 - 2.0 ** -24)
    else:
        t["rng_seeds"] = torch.randint(-2 ** 63, 2 ** 63 - 1, (B,), generator=g, device=dev)
    if case["logprobs"] >= 0:
        t["num_logprobs"] = case["logprobs"]
    return t


def _greedy_metadata():
    return SamplingMetadata(temperature=None, all_greedy=True, all_random=False, top_p=None, top_k=None,
                            generators={}, max_num_logprobs=None, no_penalties=True,
                            prompt_token_ids=None, frequency_penalties=None, presence_penalties=None,
                            repetition_penalties=None, output_token_ids=[])


def prepare(case, seed):
    t = _inputs(case, seed)
    op = case["op"]
    if op == "sample":
        call = ops.prepare_sample(t.pop("logits"), **t)
        r = call.result
        out = {"sampled": r.sampled, "num_kept": r.num_kept}
        if r.logprob_ids is not None:
            out.update(ids=r.logprob_ids, logprob=r.logprob_vals[:, 0], top=r.logprob_vals[:, 1:],
                       ranks=r.logprob_ranks)
        return {"op": op, "call": call, "out": out}
    if op == "forward":
        return {"op": op, "sampler": Sampler(), "logits": t["logits"], "metadata": _greedy_metadata()}
    return {"op": op, "logits": t["logits"], "k": case["top_k"], "temperature": t.get("temperature")}


def run(state):
    op = state["op"]
    if op == "sample":
        state["call"].launch()
        return state["out"]
    if op == "forward":
        return {"sampled": state["sampler"].forward(state["logits"], state["metadata"]).sampled_token_ids}
    if op == "softmax":
        probs, row_max, log_sum = ops.softmax(state["logits"], state["temperature"])
        return {"probs": probs, "row_max": row_max, "log_sum": log_sum}
    values, ids = ops.topk(state["logits"], state["k"])
    return {"values": values, "ids": ids}


def work(case):
    """Logits, history, masks and the row parameters read once, outputs written once.  Of the
    uniforms only those of surviving tokens are needed: they are not counted."""
    B, V = case["batch"], case["vocab"]
    size = 4 if case["dtype"] == "f32" else 2
    total = B * V * size + 4 * B
    if case["op"] == "sample":
        total += 36 * B + 4 * B * case["history"] + 8 * B * case["bans"]
        if case["allowed"]:
            total += B * V // 8
        if case["logprobs"] >= 0:
            total += B * (8 * (case["logprobs"] + 1) + 4)
    elif case["op"] == "softmax":
        total += 4 * B * V + 8 * B
    elif case["op"] == "topk":
        total += 8 * B * case["top_k"]
    return {"bytes": total, "flops": 0}


def tolerance(case):
    if case["op"] == "softmax":
        # fp32: y = x / T and y - max each round once (up to 2^-24 of their size, so about 1e-6
        # of a probability), the exponential and the product once more
        return {"rel": 1.5e-6, "max": 1e-5}
    if case["op"] == "sample" and case["logprobs"] >= 0:
        # x - logsumexp in fp32: half an ulp of the result, and of the normaliser
        return {"rel": 2e-7, "max": 1e-6}
    return "exact"


def exact(case, seed):
    """Float outputs in 64 bits; tokens and counts (whole numbers, drawn by the race) have none."""
    op = case["op"]
    if op == "forward" or (op == "sample" and case["logprobs"] < 0):
        return None
    t = _inputs(case, seed)
    x = t["logits"]
    if op == "softmax":
        y = x.double() / t["temperature"].double().unsqueeze(1)
        m = y.amax(1)
        e = torch.exp(y - m.unsqueeze(1))
        s = e.sum(1)
        return {"probs": e / s.unsqueeze(1), "row_max": m, "log_sum": s.log()}
    if op == "topk":
        return {"values": torch.topk(x.double(), case["top_k"]).values, "ids": None}
    top = []
    for rows in x.split(64):
        d = rows.double()
        top.append(torch.topk(d, case["logprobs"]).values - torch.logsumexp(d, 1, keepdim=True))
    return {"sampled": None, "num_kept": None, "ids": None, "logprob": None, "top": torch.cat(top),
            "ranks": None}
