"""Measured workloads of the Gated DeltaNet decode and prefill entry points.

Each case is one call of ``gdn_hip.gdn_decode`` or ``gdn_hip.gdn_prefill`` as a serving
program makes it. Head layouts are the two that the repository's tests and benchmark use:
16 q/k heads with 32 v heads, and 4 q/k heads with 8 v heads, head size 128. ``listed()``
gives the fixed cases, ``draw()`` more of the same ranges:

* decode, 1 to 256 sequences, one token each, new state beside the old one or in place, into
  the caller's buffers or into new ones;
* prefill, 1 to 100 packed sequences of 1 to 16384 tokens, with or without an initial state,
  int32 or int64 ``cu_seqlens``, fast-decaying or long-memory gates.
"""
import math
import os
import random
import sys

import torch

_ROOT = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                     "mlsys26-flashinfer-ai-kernel-generation-contest_amd")
if _ROOT not in sys.path:
    sys.path.insert(0, _ROOT)

from gdn_hip import gdn_decode, gdn_prefill  # noqa: E402

D = 128
# largest prefills, in token x v-head units: 16384 tokens at 8 v heads, 8192 at 32
MAX_TOKENS = {8: 16384, 32: 8192}


def _decode(name, batch, hqk, hv, inplace=False, dps=True, gates="strong"):
    return dict(name=name, kind="decode", batch=batch, hqk=hqk, hv=hv, inplace=inplace, dps=dps,
                gates=gates)


def _prefill(name, n, lo, hi, hqk, hv, len_seed=0, state=True, cu64=False, dps=True,
             gates="strong"):
    return dict(name=name, kind="prefill", n=n, lo=lo, hi=hi, len_seed=len_seed, hqk=hqk, hv=hv,
                state=state, cu64=cu64, dps=dps, gates=gates)


def listed():
    return [
        # one user's next token: launch and host latency
        _decode("decode_1", 1, 16, 32),
        # a small batch called in the simplest form, outputs allocated by the call
        _decode("decode_7_fresh", 7, 4, 8, dps=False),
        # a serving batch, the benchmark's headline: HBM stream
        _decode("decode_64", 64, 16, 32),
        # a full batch that updates its state where it stands
        _decode("decode_256_inplace", 256, 16, 32, inplace=True),
        # a short ragged prompt: one whole chunk and a part of one
        _prefill("prefill_1x77", 1, 77, 77, 4, 8, state=False),
        # an ordinary single prompt, continued from a state
        _prefill("prefill_1x300", 1, 300, 300, 16, 32),
        # a single long-memory prompt at the small head layout
        _prefill("prefill_1x1024", 1, 1024, 1024, 4, 8, gates="mild"),
        # a small ragged batch
        _prefill("prefill_8_var", 8, 64, 1024, 4, 8, len_seed=7, cu64=True),
        # the benchmark's packed batch: 16 sequences, 64 to 1024 tokens each
        _prefill("prefill_16_var", 16, 64, 1024, 16, 32),
        # the benchmark's single sequence from a zero state
        _prefill("prefill_1x4096", 1, 4096, 4096, 16, 32, state=False),
        # a long document, long memory
        _prefill("prefill_1x16384", 1, 16384, 16384, 4, 8, state=False, gates="mild"),
        # many short requests packed together
        _prefill("prefill_100_short", 100, 1, 130, 16, 32, len_seed=3),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    hqk, hv = rng.choice([(16, 32), (4, 8)])
    gates = rng.choice(["strong", "strong", "mild"])
    dps = rng.random() < 0.75
    if rng.random() < 0.4:
        c = _decode("", _log_int(rng, 1, 256), hqk, hv, inplace=dps and rng.random() < 0.4,
                    dps=dps, gates=gates)
    else:
        n = _log_int(rng, 1, 100)
        most = MAX_TOKENS[hv] // n
        hi = _log_int(rng, 24, most)
        lo = max(1, int(hi * rng.choice([0.05, 0.5, 1.0])))
        c = _prefill("", n, lo, hi, hqk, hv, len_seed=rng.randrange(1 << 20),
                     state=rng.random() < 0.7, cu64=rng.random() < 0.3, dps=dps, gates=gates)
    del c["name"]
    return c


def _lengths(case):
    r = random.Random(case["len_seed"])
    return [r.randint(case["lo"], case["hi"]) for _ in range(case["n"])]


def _inputs(case, seed):
    """q, k unit vectors, v, a, b ~ N(0, 1), dt_bias ~ U(-1, 1); strong gates A_log ~
    U(0, ln 16), mild gates U(-6, -3); state ~ N(0, 0.02^2)."""
    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev)
    g.manual_seed(int(seed))
    hqk, hv = case["hqk"], case["hv"]
    lead = (case["batch"], 1) if case["kind"] == "decode" else (sum(_lengths(case)),)
    n = case["batch"] if case["kind"] == "decode" else case["n"]

    def randn(*shape):
        return torch.randn(shape, generator=g, device=dev)

    def unit(*shape):
        x = randn(*shape)
        return (x / x.norm(dim=-1, keepdim=True)).to(torch.bfloat16)

    p = dict(q=unit(*lead, hqk, D), k=unit(*lead, hqk, D),
             v=randn(*lead, hv, D).to(torch.bfloat16),
             a=randn(*lead, hv).to(torch.bfloat16), b=randn(*lead, hv).to(torch.bfloat16))
    u = torch.rand(hv, generator=g, device=dev)
    p["A_log"] = u * math.log(16.0) if case["gates"] == "strong" else -6.0 + 3.0 * u
    p["dt_bias"] = torch.rand(hv, generator=g, device=dev) * 2.0 - 1.0
    p["state"] = randn(n, hv, D, D) * 0.02 if case.get("state", True) else None
    if case["kind"] == "prefill":
        cu = [0]
        for x in _lengths(case):
            cu.append(cu[-1] + x)
        p["cu_seqlens"] = torch.tensor(cu, device=dev, dtype=torch.int64 if case["cu64"]
                                       else torch.int32)
    return p


def prepare(case, seed):
    p = _inputs(case, seed)
    args = [p["q"], p["k"], p["v"], p["state"], p["A_log"], p["a"], p["dt_bias"], p["b"]]
    if case["kind"] == "prefill":
        args.append(p["cu_seqlens"])
    args.append(1.0 / math.sqrt(D))
    if case["dps"]:
        dev, hv = p["q"].device, case["hv"]
        n = case["batch"] if case["kind"] == "decode" else case["n"]
        args.append(torch.empty(p["v"].shape, dtype=torch.bfloat16, device=dev))
        args.append(p["state"] if case.get("inplace") else
                    torch.empty((n, hv, D, D), dtype=torch.float32, device=dev))
    return gdn_decode if case["kind"] == "decode" else gdn_prefill, args


def run(state):
    call, args = state
    return call(*args)


def work(case):
    """Bytes: every input read once, every output written once. Flops: the token recurrence
    (S k, the rank-1 update, S q), without which no form of the computation does."""
    hqk, hv = case["hqk"], case["hv"]
    if case["kind"] == "decode":
        tokens = n = case["batch"]
    else:
        tokens, n = sum(_lengths(case)), case["n"]
    state = n * hv * D * D * 4 * (2 if case.get("state", True) else 1)
    per_token = 2 * hqk * D * 2 + 2 * hv * D * 2 + 2 * hv * 2
    return {"bytes": tokens * per_token + state + 2 * hv * 4,
            "flops": tokens * hv * 6 * D * D}


def tolerance(case):
    """Outputs are bf16. A decode rounds once: a relative 2-norm of 1.7e-3 against 64 bits, at
    most 3.9e-3 of an element.
    A prefill's readout products take bf16 operands too: 2.9e-3, at most
    4.6e-2 of the root mean square."""
    return {"rel": 6e-3, "max": 0.016} if case["kind"] == "decode" else {"rel": 1.2e-2, "max": 0.2}


def exact(case, seed):
    """The token recurrence in float64."""
    p = _inputs(case, seed)
    hqk, hv = case["hqk"], case["hv"]
    if case["kind"] == "decode":
        lens, flat = [1] * case["batch"], {x: p[x].squeeze(1) for x in "qkvab"}
    else:
        lens, flat = _lengths(case), {x: p[x] for x in "qkvab"}
    dev = p["q"].device
    n = len(lens)
    order = sorted(range(n), key=lambda i: -lens[i])
    at = torch.tensor([sum(lens[:i]) for i in range(n)], device=dev)[order]
    S = torch.zeros(n, hv, D, D, dtype=torch.float64, device=dev)
    if p["state"] is not None:
        S.copy_(p["state"][order])
    x = flat["a"].double() + p["dt_bias"].double()
    alpha = torch.exp(-torch.exp(p["A_log"].double()) * torch.nn.functional.softplus(x))
    beta = torch.sigmoid(flat["b"].double())
    scale = 1.0 / math.sqrt(D)
    out = torch.zeros(flat["v"].shape, dtype=torch.float64, device=dev)
    live = n
    for t in range(max(lens)):
        while lens[order[live - 1]] <= t:
            live -= 1
        row = at[:live] + t
        k = flat["k"][row].double().repeat_interleave(hv // hqk, 1)[:, :, None, :]
        q = flat["q"][row].double().repeat_interleave(hv // hqk, 1)[:, :, None, :]
        s = S[:live]
        s *= alpha[row][:, :, None, None]
        d = beta[row][:, :, None] * (flat["v"][row].double() - (s * k).sum(-1))
        s += d[..., None] * k
        out[row] = scale * (s * q).sum(-1)
    new_state = torch.empty_like(S)
    new_state[order] = S
    return out.reshape(p["v"].shape), new_state
