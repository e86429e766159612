"""The calls whose time this repository is judged by: GDN decode steps and varlen prefills.

Each case is one pass through a public entry point (``decode.launch_gdn``,
``prefill.launch_gdn``, or the replay of a HIP graph that captured decode
steps), on inputs made from a seed on the GPU:

* q, k: unit rows (L2-normalised over the head dim), bf16; v, a, b: randn, bf16;
* state: 0.02 randn, fp32 (a state carried from earlier tokens), or none;
* gates by ``decay``:
  - "fast": A_log U(-1, 1), dt_bias 0.1 randn (the benchmark's gates: a head
    forgets within a few dozen tokens);
  - "mixed": A_log = log U(1, 16), dt_bias = softplus^-1 of a step that is
    log-uniform in [0.001, 0.1] (the usual initialisation of gated delta
    layers: some heads forget within a chunk, some hold for thousands of tokens);
  - "slow": A_log U(-8, -5), dt_bias 0.1 randn (every head holds for long).

``draw`` gives further cases of the same ranges: decode batches of 1 to 256,
graphs of 4 to 28 layers with batches of 1 to 16, prefills of 1 to 512
sequences with 1 to 32768 tokens in all, every gate regime, with and without
an initial state, 32- and 64-bit cu_seqlens, own and kept workspaces.
"""

from __future__ import annotations

import math
import random

import torch

from kachua_mlsys_amd import decode, prefill

HQ, HV, D = 4, 8, 128
SCALE = 1.0 / math.sqrt(D)


def _decode(batch, decay="fast", **kw):
    return {"op": "decode", "batch": batch, "decay": decay, **kw}


def _graph(layers, batch, decay="mixed", **kw):
    return {"op": "graph", "layers": layers, "batch": batch, "decay": decay, **kw}


def _prefill(seqs, tokens, lo, hi, decay="fast", state=True, cu=32, workspace=False, **kw):
    return {"op": "prefill", "seqs": seqs, "tokens": tokens, "lo": lo, "hi": hi, "decay": decay,
            "state": state, "cu": cu, "workspace": workspace, **kw}


def listed():
    return [
        # one user's next token, eager: what a single-stream chat pays per layer
        _decode(1, name="decode_1"),
        # the reference's largest decode batch, and this repository's headline
        _decode(64, name="decode_64"),
        # a large serving batch: nothing but state traffic
        _decode(256, "mixed", name="decode_256"),
        # a small batch's decode step over all gated-delta layers of a model,
        # captured once and replayed per token, as serving engines run it
        _graph(24, 4, name="decode_graph_24x4"),
        # the shortest prompts, or a speculative window: latency of one call
        _prefill(1, 16, 16, 16, name="prefill_1x16"),
        # a handful of short prompts admitted in one scheduler step
        _prefill(8, 403, 9, 90, "mixed", name="prefill_8x50"),
        # a first prompt without history
        _prefill(1, 1024, 1024, 1024, state=False, name="prefill_1x1024"),
        # a scheduler step over many medium prompts; torch's default index type
        _prefill(32, 8192, 32, 1500, "mixed", cu=64, name="prefill_32x256"),
        # the benchmark's varlen batch (16 sequences, 16,384 tokens)
        _prefill(16, 16384, 128, 4096, name="prefill_16x1024"),
        # the same lengths under gates that hold for long
        _prefill(16, 16384, 128, 4096, "slow", name="prefill_16x1024_slow"),
        # the benchmark's batch of many short sequences (continued chats)
        _prefill(512, 17408, 4, 64, name="prefill_512x34"),
        # one long document, workspace kept by the program
        _prefill(1, 32768, 32768, 32768, "mixed", workspace=True, name="prefill_1x32768"),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    decay = rng.choice(["fast", "mixed", "slow"])
    op = rng.choice(["decode", "graph", "prefill", "prefill", "prefill"])
    if op == "decode":
        return _decode(_logint(rng, 1, 256), decay)
    if op == "graph":
        return _graph(rng.randint(4, 28), _logint(rng, 1, 16), decay)
    seqs = _logint(rng, 1, 512)
    # at least a token a sequence on average; many-sequence batches hold
    # shorter sequences, so that no draw costs more than the listed cases
    top = min(24576 if decay == "slow" else 32768, 40 * (832 - seqs))
    tokens = _logint(rng, max(8, 3 * seqs), max(top, 3 * seqs))
    mean = tokens / seqs
    lo = max(1, int(mean / rng.choice([1.0, 4.0, 8.0])))
    hi = max(lo, int(mean * rng.choice([1.0, 2.0, 4.0])))
    return _prefill(seqs, tokens, lo, hi, decay, state=rng.random() < 0.75, cu=rng.choice([32, 64]),
                    workspace=rng.random() < 0.3)


def _lengths(case):
    """seqs lengths, log-uniform in [lo, hi], scaled to sum to tokens (each at least 1)."""
    n, total = case["seqs"], case["tokens"]
    rng = random.Random(1000003 * n + total)
    raw = [math.exp(rng.uniform(math.log(case["lo"]), math.log(case["hi"]))) for _ in range(n)]
    f = total / sum(raw)
    got = [max(1, int(x * f)) for x in raw]
    i = 0
    while sum(got) != total:   # the rounding's rest, spread over the sequences
        step = 1 if sum(got) < total else -1
        if got[i % n] + step >= 1:
            got[i % n] += step
        i += 1
    return got


def _unit(shape, g):
    x = torch.randn(shape, generator=g, device="cuda")
    return (x / x.norm(dim=-1, keepdim=True)).to(torch.bfloat16)


def _gates(decay, g):
    def u(lo, hi):
        return torch.rand(HV, generator=g, device="cuda") * (hi - lo) + lo

    if decay == "mixed":
        A_log = torch.log(u(1.0, 16.0))
        dt = torch.exp(u(math.log(1e-3), math.log(1e-1)))
        return A_log, dt + torch.log(-torch.expm1(-dt))
    dt_bias = 0.1 * torch.randn(HV, generator=g, device="cuda")
    return (u(-1.0, 1.0) if decay == "fast" else u(-8.0, -5.0)), dt_bias


def _decode_inputs(batch, decay, g):
    def bf(*shape):
        return torch.randn(shape, generator=g, device="cuda").to(torch.bfloat16)

    A_log, dt_bias = _gates(decay, g)
    return {"q": _unit((batch, 1, HQ, D), g), "k": _unit((batch, 1, HQ, D), g), "v": bf(batch, 1, HV, D),
            "state": 0.02 * torch.randn((batch, HV, D, D), generator=g, device="cuda"),
            "A_log": A_log, "a": bf(batch, 1, HV), "dt_bias": dt_bias, "b": bf(batch, 1, HV)}


def _prefill_inputs(case, g):
    def bf(*shape):
        return torch.randn(shape, generator=g, device="cuda").to(torch.bfloat16)

    T, n = case["tokens"], case["seqs"]
    A_log, dt_bias = _gates(case["decay"], g)
    cu = [0]
    for x in _lengths(case):
        cu.append(cu[-1] + x)
    return {"q": _unit((T, HQ, D), g), "k": _unit((T, HQ, D), g), "v": bf(T, HV, D),
            "state": 0.02 * torch.randn((n, HV, D, D), generator=g, device="cuda") if case["state"] else None,
            "A_log": A_log, "a": bf(T, HV), "dt_bias": dt_bias, "b": bf(T, HV),
            "cu_seqlens": torch.tensor(cu, dtype=torch.int32 if case["cu"] == 32 else torch.int64, device="cuda")}


def _all_inputs(case, seed):
    g = torch.Generator("cuda").manual_seed(seed)
    if case["op"] == "prefill":
        return [_prefill_inputs(case, g)]
    return [_decode_inputs(case["batch"], case["decay"], g) for _ in range(case.get("layers", 1))]


def _step(s):
    return decode.launch_gdn(s["q"], s["k"], s["v"], s["state"], s["A_log"], s["a"], s["dt_bias"], s["b"], SCALE,
                             s["out"], s["new_state"])


def prepare(case, seed):
    sets = _all_inputs(case, seed)
    for s in sets:
        if case["op"] == "prefill":
            s["out"] = torch.empty_like(s["v"])
            s["new_state"] = torch.empty((case["seqs"], HV, D, D), device="cuda")
            s["workspace"] = None
            if case["workspace"]:
                need = prefill.workspace_bytes(case["seqs"], case["tokens"])
                s["workspace"] = torch.empty(need, dtype=torch.uint8, device="cuda")
        else:
            s["out"] = torch.empty((case["batch"], HV, D), dtype=torch.bfloat16, device="cuda")
            s["new_state"] = torch.empty_like(s["state"])
    st = {"op": case["op"], "sets": sets}
    if case["op"] == "graph":
        for s in sets:
            _step(s)
        torch.cuda.synchronize()
        st["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(st["graph"]):
            for s in sets:
                _step(s)
    return st


def run(st):
    if st["op"] == "graph":
        st["graph"].replay()
        return [(s["out"], s["new_state"]) for s in st["sets"]]
    s = st["sets"][0]
    if st["op"] == "decode":
        return _step(s)
    return prefill.launch_gdn(s["q"], s["k"], s["v"], s["state"], s["A_log"], s["a"], s["dt_bias"], s["b"],
                              s["cu_seqlens"], SCALE, s["out"], s["new_state"], workspace=s["workspace"])


def work(case):
    """Inputs read once, outputs written once; the token recurrence's three
    128 x 128 products per v-head and token (S k, the rank-1 update, S q)."""
    if case["op"] == "prefill":
        tokens, seqs, layers = case["tokens"], case["seqs"], 1
        states = seqs * (2 if case["state"] else 1)
        index = (seqs + 1) * case["cu"] // 8
    else:
        tokens, layers, index = case["batch"], case.get("layers", 1), 0
        states = 2 * tokens
    per_token = 2 * HQ * D * 2 + 2 * HV * D * 2 + 2 * HV * 2   # q, k; v, out; a, b
    return {"bytes": layers * (states * HV * D * D * 4 + tokens * per_token + 2 * HV * 4 + index),
            "flops": layers * tokens * HV * 3 * 2 * D * D}


def tolerance(case):
    """bf16 outputs of fp32 sums; prefills form their chunks' terms in 16-bit operands besides."""
    if case["op"] == "prefill":
        return {"rel": 1.2e-2, "max": 0.1}
    return {"rel": 8e-3, "max": 0.06}


def _recur(S, q, k, v, g, beta):
    """One token of every sequence in S [n, 8, 128, 128] (updated in place) -> outputs [n, 8, 128]."""
    k, q = k.repeat_interleave(HV // HQ, 1), q.repeat_interleave(HV // HQ, 1)
    S.mul_(g[..., None, None])
    delta = beta[..., None] * (v - (S * k[..., None, :]).sum(-1))
    S.addcmul_(delta[..., None], k[..., None, :])
    return SCALE * (S * q[..., None, :]).sum(-1)


def _gate64(s):
    x = s["a"].double() + s["dt_bias"].double()
    return torch.exp(-torch.exp(s["A_log"].double()) * torch.nn.functional.softplus(x)), torch.sigmoid(s["b"].double())


def exact(case, seed):
    """The token recurrence in 64 bits."""
    got = []
    for s in _all_inputs(case, seed):
        g, beta = _gate64(s)
        q, k, v = s["q"].double(), s["k"].double(), s["v"].double()
        if case["op"] != "prefill":
            S = s["state"].double()
            got.append((_recur(S, q[:, 0], k[:, 0], v[:, 0], g[:, 0], beta[:, 0]), S))
            continue
        lens = _lengths(case)
        order = sorted(range(len(lens)), key=lambda i: -lens[i])   # longest first: the running ones are a prefix
        start = torch.tensor([sum(lens[:i]) for i in order], device="cuda")
        n = case["seqs"]
        S = (s["state"][order].double() if case["state"]
             else torch.zeros((n, HV, D, D), dtype=torch.float64, device="cuda"))
        out = torch.empty((case["tokens"], HV, D), dtype=torch.float64, device="cuda")
        run_, live = n, [lens[i] for i in order]
        for t in range(live[0]):
            while live[run_ - 1] <= t:
                run_ -= 1
            at = start[:run_] + t
            out[at] = _recur(S[:run_], q[at], k[at], v[at], g[at], beta[at])
        back = torch.empty_like(S)
        back[torch.tensor(order, device="cuda")] = S
        got.append((out, back))
    return got if case["op"] == "graph" else got[0]
