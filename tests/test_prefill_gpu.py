"""GPU parity of gdn_prefill (HIP, chunked WY form) against the float64 CPU oracle.

Bars (gdn_hip.parity): output bf16 atol = rtol = 1e-2 (both-condition rule of
FAQ.md:104-110); new_state fp32 elementwise rtol = 1e-3 / atol = 1e-4 and normwise
relative error <= 1e-3.
"""
import ctypes

import numpy as np
import pytest
import torch

from gdn_hip import _lib, gdn_decode, gdn_prefill, release_workspace
from gdn_hip.inputs import prefill_inputs, varlen_lengths, with_extreme_gates
from gdn_hip.parity import check_output, check_state
from oracle import gdn_oracle as O

pytestmark = pytest.mark.gpu


def _oracle(inp):
    return O.prefill(inp.q, inp.k, inp.v, inp.state, inp.A_log, inp.a, inp.dt_bias, inp.b,
                     inp.cu_seqlens, inp.scale)


def _check(out, ns, ref_out, ref_ns, label):
    vo = check_output(out, ref_out)
    vs = check_state(ns, ref_ns)
    print(f"[{label}] output {vo} | state {vs}", flush=True)
    assert vo.ok, f"{label}: output {vo}"
    assert vs.ok, f"{label}: new_state {vs}"


def _run(dev, inp, label, **kw):
    print(f"[{label}] launching T={inp.q.shape[0]} lens={inp.seqlens[:8]}...", flush=True)
    ref_out, ref_ns = _oracle(inp)
    g = inp.to(dev)
    out, ns = gdn_prefill(*g.args(), **kw)
    torch.cuda.synchronize()
    _check(out, ns, ref_out, ref_ns, label)
    return g, out, ns


@pytest.mark.parametrize("lens", [[1], [5], [63], [64], [65], [128], [129], [200, 37]])
def test_prefill_small(dev, lens):
    _run(dev, prefill_inputs(lens, seed=len(lens) * 100 + lens[0], with_state=True),
         f"lens={lens}")


def test_prefill_single_4k_zero_state(dev):
    """One 4096-token sequence, zero initial state (state=None)."""
    _run(dev, prefill_inputs([4096], seed=3, with_state=False), "4k state=None")


def test_prefill_varlen_16(dev):
    """16 sequences, lengths ~U[64,1024] from the seed, non-zero fp32 initial state."""
    lens = varlen_lengths(16, seed=0)
    _run(dev, prefill_inputs(lens, seed=0, with_state=True), "varlen16")


@pytest.mark.parametrize("gates", ["mild", "none"])
def test_prefill_long_memory_gates(dev, gates):
    """alpha ~ 0.99 or exactly 1: the state carries across many chunks."""
    _run(dev, prefill_inputs([300, 700, 64], seed=5, with_state=True, gates=gates,
                             state_std=0.1), f"gates={gates}")


@pytest.mark.parametrize("hqk,hv", [(4, 8), (8, 8), (2, 8), (1, 4), (2, 6), (1, 3)])
def test_prefill_head_layouts(dev, hqk, hv):
    _run(dev, prefill_inputs([150, 90, 257], hqk=hqk, hv=hv, seed=9, with_state=True),
         f"hqk={hqk} hv={hv}")


def test_prefill_empty_sequences_and_gaps(dev):
    """Zero-length sequences keep their state; tokens outside every sequence read as
    zero output (gdn_prefill/solution/triton/kernel.py:286)."""
    _run(dev, prefill_inputs([0, 70, 0, 0, 130, 0], seed=17, with_state=True, pad_tokens=45),
         "empty+gaps")


@pytest.mark.parametrize("scale", [None, 0.0, 0.25, "host tensor", "device tensor"])
def test_prefill_scale_defaults(dev, scale):
    """scale None / 0 -> 1/sqrt(D) (gdn_prefill/solution/triton/kernel.py:276-277); a
    one-element tensor is read as its value (0.25 here). Through the Python path (no
    destination buffers), destination-passing calls (the C++ fast path for a float or None
    scale, the Python path for a tensor) and the fast path called directly, each against
    the oracle."""
    inp = prefill_inputs([150, 64, 1], hqk=4, hv=8, seed=31, with_state=True)
    inp.scale = 0.25 if isinstance(scale, str) else scale
    ref_o, ref_s = _oracle(inp)
    g = inp.to(dev)
    args = list(g.args())
    if isinstance(scale, str):
        args[-1] = torch.tensor([0.25], device=dev if scale == "device tensor" else "cpu")
    T, N = g.q.shape[0], len(inp.seqlens)
    out, ns = gdn_prefill(*args)
    o2 = torch.empty((T, 8, 128), dtype=torch.bfloat16, device=dev)
    n2 = torch.empty((N, 8, 128, 128), dtype=torch.float32, device=dev)
    gdn_prefill(*args, output=o2, new_state=n2)
    torch.cuda.synchronize()
    _check(out, ns, ref_o, ref_s, f"scale={scale}")
    _check(o2, n2, ref_o, ref_s, f"scale={scale} destination-passing")
    if not isinstance(scale, str):
        o3, n3 = torch.empty_like(o2), torch.empty_like(n2)
        assert _lib.fast().prefill(*args[:-1], 0.0 if scale is None else scale, o3, n3, 0) == 0
        torch.cuda.synchronize()
        assert torch.equal(o3, out) and torch.equal(n3, ns)


def test_prefill_int64_cu_seqlens(dev):
    _run(dev, prefill_inputs([99, 1, 250], seed=19, with_state=True, cu_dtype=torch.int64),
         "cu int64")


def test_prefill_inplace_state(dev):
    inp = prefill_inputs([180, 75], seed=23, with_state=True)
    ref_out, ref_ns = _oracle(inp)
    g = inp.to(dev)
    out, ns = gdn_prefill(*g.args(), new_state=g.state)
    torch.cuda.synchronize()
    assert ns.data_ptr() == g.state.data_ptr()
    _check(out, ns, ref_out, ref_ns, "in-place")


def test_prefill_explicit_zero_state_equals_none(dev):
    inp = prefill_inputs([333], seed=29, with_state=False).to(dev)
    o1, s1 = gdn_prefill(*inp.args())
    z = torch.zeros((1, 32, 128, 128), dtype=torch.float32, device=dev)
    args = list(inp.args())
    args[3] = z
    o2, s2 = gdn_prefill(*args)
    torch.cuda.synchronize()
    assert torch.equal(o1, o2) and torch.equal(s1, s2)


def test_prefill_strided_and_preallocated(dev):
    """q/k/v as views of a fused projection; preallocated (poisoned) outputs."""
    inp = prefill_inputs([77, 160], seed=31, with_state=True)
    ref_out, ref_ns = _oracle(inp)
    g = inp.to(dev)
    T = g.q.shape[0]
    qkv = torch.empty((T, 16 + 16 + 32, 128), dtype=torch.bfloat16, device=dev)
    qkv[:, :16], qkv[:, 16:32], qkv[:, 32:] = g.q, g.k, g.v
    out = torch.full((T, 32, 128), 7.0, dtype=torch.bfloat16, device=dev)
    ns = torch.full_like(g.state, 7.0)
    o, s = gdn_prefill(qkv[:, :16], qkv[:, 16:32], qkv[:, 32:], g.state, g.A_log, g.a,
                       g.dt_bias, g.b, g.cu_seqlens, g.scale, output=out, new_state=ns)
    torch.cuda.synchronize()
    assert o.data_ptr() == out.data_ptr() and s.data_ptr() == ns.data_ptr()
    _check(o, s, ref_out, ref_ns, "strided")


def test_prefill_deterministic(dev):
    inp = prefill_inputs(varlen_lengths(8, seed=4), seed=4, with_state=True).to(dev)
    o1, s1 = gdn_prefill(*inp.args())
    o2, s2 = gdn_prefill(*inp.args())
    torch.cuda.synchronize()
    assert torch.equal(o1, o2) and torch.equal(s1, s2)


def test_prefill_no_sequences_and_no_tokens(dev):
    inp = prefill_inputs([], seed=1, with_state=True, pad_tokens=10).to(dev)
    out, ns = gdn_prefill(*inp.args())
    torch.cuda.synchronize()
    assert out.shape == (10, 32, 128) and torch.all(out == 0)
    assert ns.shape == (0, 32, 128, 128)
    inp = prefill_inputs([0, 0], seed=2, with_state=True).to(dev)
    out, ns = gdn_prefill(*inp.args())
    torch.cuda.synchronize()
    assert out.shape == (0, 32, 128) and torch.equal(ns, inp.state)


def test_prefill_resume_split(dev):
    """prefill(x[:m]) then prefill(x[m:], state) against the oracle's prefill(x): the
    state handoff between calls (k-last new_state fed back as state,
    gdn_prefill/solution/triton/kernel.py:32,288-299)."""
    inp = prefill_inputs([500], seed=37, with_state=True, gates="mild")
    ref_o, ref_s = _oracle(inp)
    g = inp.to(dev)
    m = 203
    cu1 = torch.tensor([0, m], dtype=torch.int32, device=dev)
    cu2 = torch.tensor([0, 500 - m], dtype=torch.int32, device=dev)
    o1, s1 = gdn_prefill(g.q[:m], g.k[:m], g.v[:m], g.state, g.A_log, g.a[:m],
                         g.dt_bias, g.b[:m], cu1, g.scale)
    o2, s2 = gdn_prefill(g.q[m:], g.k[m:], g.v[m:], s1, g.A_log, g.a[m:],
                         g.dt_bias, g.b[m:], cu2, g.scale)
    torch.cuda.synchronize()
    _check(torch.cat([o1, o2]), s2, ref_o, ref_s, "resume vs oracle")


def test_prefill_records_past_2gib(dev):
    """Maximum sizes: one 327,680-token sequence at 32 v-heads, whose workspace records
    (5,121 chunks x 32 v-heads x 16 KB = 2.7 GB) reach past 2^31 bytes, against the same
    sequence prefilled as five chained 65,536-token calls (0.5 GB of records each, the
    state handed from call to call). The two runs plan and cut the sequence differently,
    so they agree to rounding; an offset truncated to 32 bits in the large run would read
    or write the wrong records. Inputs are drawn on the GPU and compared there (the oracle
    would need ~0.7 TFLOP in fp64); mild decay keeps earlier chunks' states significant."""
    T, piece, hqk, hv = 5 << 16, 1 << 16, 2, 32
    g = torch.Generator(device=dev)
    g.manual_seed(61)
    unit = lambda *s: torch.nn.functional.normalize(  # noqa: E731
        torch.randn(*s, generator=g, device=dev), dim=-1).to(torch.bfloat16)
    q, k = unit(T, hqk, 128), unit(T, hqk, 128)
    v = torch.randn(T, hv, 128, generator=g, device=dev).to(torch.bfloat16)
    a = torch.randn(T, hv, generator=g, device=dev).to(torch.bfloat16)
    b = torch.randn(T, hv, generator=g, device=dev).to(torch.bfloat16)
    A_log = -6.0 + 3.0 * torch.rand(hv, generator=g, device=dev)
    dt_bias = torch.rand(hv, generator=g, device=dev) * 2.0 - 1.0
    state = torch.randn(1, hv, 128, 128, generator=g, device=dev) * 0.05
    scale = 128 ** -0.5
    ws = _lib.load().gdn_prefill_workspace_size(T, 1, hqk, hv, 128)
    print(f"[{T} tokens] whole-sequence run, workspace {ws / 2**30:.2f} GiB", flush=True)
    assert ws > (1 << 31)
    cu = torch.tensor([0, T], dtype=torch.int32, device=dev)
    o_full, s_full = gdn_prefill(q, k, v, state, A_log, a, dt_bias, b, cu, scale)
    torch.cuda.synchronize()
    cu_p = torch.tensor([0, piece], dtype=torch.int32, device=dev)
    s = state
    outs = []
    for i in range(T // piece):
        sl = slice(i * piece, (i + 1) * piece)
        o, s = gdn_prefill(q[sl], k[sl], v[sl], s, A_log, a[sl], dt_bias, b[sl], cu_p, scale)
        outs.append(o)
    torch.cuda.synchronize()
    # the output bar of gdn_hip.parity (both-condition rule), evaluated on the device
    x, y = o_full.float(), torch.cat(outs).float()
    d = (x - y).abs()
    nfail = int(((d > 1e-2) & (d > 1e-2 * y.abs())).sum())
    vs = check_state(s_full, s)
    print(f"[{T} tokens] whole vs chained: output max_abs={float(d.max()):.3e} fail={nfail} | "
          f"state {vs}", flush=True)
    assert nfail == 0 and torch.isfinite(x).all()
    assert vs.ok
    del x, y, d, o_full, outs, q, k, v
    release_workspace()


@pytest.mark.parametrize("gates", ["strong", "mild"])
def test_prefill_then_decode_matches_oracle(dev, gates):
    """Prefill's new_state feeds decode in the same k-last layout
    (gdn_prefill/solution/triton/kernel.py:32, gdn_decode/solution/triton/kernel.py:8,17):
    prefill(x) followed by four decode steps t1..t4 must equal the oracle's prefill of
    x || t1..t4, token by token and in the final state, for two sequences at once."""
    L, n_dec = [257, 64], 4
    inp = prefill_inputs([x + n_dec for x in L], seed=41, with_state=True, gates=gates)
    ref_o, ref_s = _oracle(inp)
    g = inp.to(dev)
    cu = inp.cu_seqlens.tolist()
    # prefill of the first L[i] tokens of each sequence, packed
    idx = torch.cat([torch.arange(cu[i], cu[i] + L[i]) for i in range(2)]).to(dev)
    cu_p = torch.tensor([0, L[0], L[0] + L[1]], dtype=torch.int32, device=dev)
    o_p, s = gdn_prefill(g.q[idx], g.k[idx], g.v[idx], g.state, g.A_log, g.a[idx],
                         g.dt_bias, g.b[idx], cu_p, g.scale)
    outs = []
    for j in range(n_dec):
        t = torch.tensor([cu[i] + L[i] + j for i in range(2)], device=dev)
        od, s = gdn_decode(g.q[t].unsqueeze(1), g.k[t].unsqueeze(1), g.v[t].unsqueeze(1), s,
                           g.A_log, g.a[t].unsqueeze(1), g.dt_bias, g.b[t].unsqueeze(1),
                           g.scale)
        outs.append(od[:, 0])
    torch.cuda.synchronize()
    vo = check_output(o_p, ref_o[idx.cpu().numpy()])
    print(f"[prefill part {gates}] output {vo}", flush=True)
    assert vo.ok
    dec_ref = np.stack([ref_o[[cu[i] + L[i] + j for i in range(2)]] for j in range(n_dec)],
                       axis=1)
    _check(torch.stack(outs, dim=1), s, dec_ref, ref_s, f"prefill->decode x{n_dec} {gates}")


def test_prefill_matches_exact_fixture(dev):
    """HIP prefill vs the rational-arithmetic known answers (tests/golden/make_golden.py)."""
    import os

    import numpy as np

    f = np.load(os.path.join(os.path.dirname(__file__), "golden", "gdn_kat_d128.npz"))

    def bf(x):
        return torch.from_numpy(x.view(np.int16).copy()).view(torch.bfloat16).to(dev)

    out, ns = gdn_prefill(bf(f["q"]), bf(f["k"]), bf(f["v"]), torch.from_numpy(f["state"]).to(dev),
                          torch.from_numpy(f["A_log"]).to(dev), bf(f["a"]),
                          torch.from_numpy(f["dt_bias"]).to(dev), bf(f["b"]),
                          torch.from_numpy(f["cu_seqlens"]).to(dev), float(f["scale"]))
    torch.cuda.synchronize()
    _check(out, ns, f["out"], f["new_state"], "exact fixture")


@pytest.mark.parametrize("nseq", [64, 65, 255, 300, 600])
def test_prefill_many_sequences(dev, nseq):
    """Many short and empty sequences. Up to 126 the prep kernel plans for itself (one
    sequence per lane up to 64, two above); from 127 the planning kernel's chunk table and
    longest-first order (its sort covers up to 512 sequences) drive prep and scan."""
    g = torch.Generator().manual_seed(nseq)
    lens = [int(x) for x in torch.randint(0, 90, (nseq,), generator=g)]
    _run(dev, prefill_inputs(lens, hqk=4, hv=8, seed=nseq, with_state=True), f"N={nseq}")


@pytest.mark.parametrize("lens,hqk,hv,state,gates", [
    # four workgroups per v-head on the column-split bodies: up to one per CU (64 pairs at
    # 256 CUs), and just above; whole sequences, segments with 0 to 3 chain steps, empty and
    # 1-token sequences, chunk edges, an odd head ratio
    ([1, 64, 65, 0, 127, 128, 129, 200], 4, 8, True, "mild"),
    ([1, 64, 65, 0, 127, 128, 129, 200, 31], 4, 8, True, "mild"),
    ([300, 65], 16, 32, False, "none"),
    ([900, 1], 4, 8, True, "none"),
    ([1500], 4, 8, True, "mild"),
    ([1600], 1, 3, True, "mild"),
    ([63], 16, 32, True, "strong"),
])
def test_prefill_column_split_scan(dev, lens, hqk, hv, state, gates):
    _run(dev, prefill_inputs(lens, hqk=hqk, hv=hv, seed=sum(lens) % 89, with_state=state,
                             gates=gates), f"column split {lens[:3]} x {hv}")


@pytest.mark.parametrize("lens,hqk,hv,state,gates", [
    # the scan with two workgroups per CU (768 (sequence, v-head) pairs and more): chunk edges
    # and remainders, empty sequences, odd and even chunk counts, the smallest batch it takes
    ([1, 63, 64, 65, 0, 127, 128, 129, 191, 192, 193, 257, 31, 2, 320, 16, 17, 96, 64, 33, 5, 48,
      80, 15], 16, 32, True, "mild"),
    ([64] * 24, 16, 32, False, "strong"),
    ([7 + 3 * i for i in range(96)], 4, 8, True, "none"),
    ([40, 0, 130] * 43, 2, 6, True, "mild"),
])
def test_prefill_wide_scan(dev, lens, hqk, hv, state, gates):
    _run(dev, prefill_inputs(lens, hqk=hqk, hv=hv, seed=sum(lens) % 97, with_state=state,
                             gates=gates), f"wide scan {len(lens)} x {hv}")


def _run_with_header(dev, inp, label, ints=16, inplace=False):
    """One prefill through the C entry point against the oracle; returns the first ints of
    the workspace header, where the planner leaves its job counts (cleared before: a call that
    plans none leaves zeros)."""
    from gdn_hip.api import _prefill_marshal
    ref_out, ref_ns = _oracle(inp)
    g = inp.to(dev)
    hv = g.v.shape[1]
    out = torch.empty(g.v.shape, dtype=torch.bfloat16, device=dev)
    ns = g.state if inplace else torch.empty((len(inp.seqlens), hv, 128, 128),
                                             dtype=torch.float32, device=dev)
    P, _, _, copy_back, keep, stream = _prefill_marshal(*g.args(), out, ns)
    assert not copy_back
    keep[-1][:4 * ints].zero_()
    print(f"[{label}] launching", flush=True)
    rc = _lib.load().gdn_prefill_launch(ctypes.byref(P), ctypes.c_void_p(stream.cuda_stream))
    assert rc == 0, _lib.load().gdn_last_error()
    torch.cuda.synchronize()
    header = keep[-1][:4 * ints].view(torch.int32).cpu().tolist()
    print(f"[{label}] header {header}", flush=True)
    _check(out, ns, ref_out, ref_ns, label)
    return header


@pytest.mark.parametrize("lens,hqk,hv,wide", [
    ([64] * 96, 4, 8, True),
    ([1500] + [40] * 95, 4, 8, False),              # a long prompt among short ones
    ([900, 0, 700] + [33] * 127, 2, 6, False),      # the same through the plan kernel
    ([20] * 519 + [600], 1, 2, False),              # too many to sort: the long one comes last
    ([20] * 520, 1, 2, True),
])
def test_prefill_wide_scan_choice(dev, lens, hqk, hv, wide):
    """768 (sequence, v-head) pairs and more, short on average: the planner gives the sequences
    to the wide scan (header[6]) unless the longest one's chain alone would take longer there
    than the whole batch in the 8-wave scan (header[5]), whose job queues then hand out every
    job once."""
    inp = prefill_inputs(lens, hqk=hqk, hv=hv, seed=len(lens), with_state=True, gates="mild")
    header = _run_with_header(dev, inp, f"wide choice N={len(lens)}")
    n = len(lens)
    assert (header[5], header[6]) == ((0, n) if wide else (n, 0))


@pytest.mark.parametrize("skewed", [False, True])
def test_prefill_wide_scan_layouts(dev, skewed):
    """768 pairs, in the wide scan and (one long sequence) in the queued 8-wave scan behind it:
    q / k / v as views of a fused projection, the output a view of a wider tensor, the state
    strided and updated in place, tokens before the first and after the last sequence."""
    lens = [1 + (37 * i) % 130 for i in range(96)]
    if skewed:
        lens[40] = 1900
    inp = prefill_inputs(lens, hqk=4, hv=8, seed=17, with_state=True, gates="mild", pad_tokens=9)
    inp.cu_seqlens = inp.cu_seqlens + 4
    ref_out, ref_ns = _oracle(inp)
    g = inp.to(dev)
    T = g.q.shape[0]
    qkv = torch.cat([g.q, g.k, g.v], dim=1)
    big = torch.full((T, 12, 128), 7.0, dtype=torch.bfloat16, device=dev)
    st = torch.full((96, 11, 128, 132), 3.0, dtype=torch.float32, device=dev)
    st[:, 2:10, :, :128] = g.state
    state, out = st[:, 2:10, :, :128], big[:, 3:11]
    print(f"[wide layouts skewed={skewed}] launching", flush=True)
    o, ns = gdn_prefill(qkv[:, :4], qkv[:, 4:8], qkv[:, 8:], state, g.A_log, g.a, g.dt_bias, g.b,
                        g.cu_seqlens, g.scale, output=out, new_state=state)
    torch.cuda.synchronize()
    assert o.data_ptr() == out.data_ptr() and ns.data_ptr() == state.data_ptr()
    _check(o, ns, ref_out, ref_ns, f"wide layouts skewed={skewed}")
    assert not out[:4].any() and not out[-5:].any()
    assert torch.all(big[:, :3] == 7) and torch.all(big[:, 11:] == 7)
    st[:, 2:10, :, :128] = 3.0
    assert torch.all(st == 3)


@pytest.mark.parametrize("cu_dtype", [torch.int32, torch.int64])
def test_prefill_planners_agree(dev, cu_dtype):
    """The prep kernel's own planning (126 sequences) and the plan kernel (the same and an empty
    one) give equal bits: empty sequences, chunk edges, a first entry below 0 and last ones past
    the end, which both clamp."""
    lens = [(0, 1, 64, 65, 130, 20)[i % 6] for i in range(126)]
    g = prefill_inputs(lens, hqk=2, hv=4, seed=5, with_state=True, gates="mild",
                       cu_dtype=cu_dtype).to(dev)
    cu = g.cu_seqlens.clone()
    cu[0] = -7
    cu[-3:] = g.q.shape[0] + 1000
    rest = (g.A_log, g.a, g.dt_bias, g.b)
    o1, s1 = gdn_prefill(g.q, g.k, g.v, g.state, *rest, cu, g.scale)
    o2, s2 = gdn_prefill(g.q, g.k, g.v, torch.cat([g.state, g.state[:1]]), *rest,
                         torch.cat([cu, cu[-1:]]), g.scale)
    torch.cuda.synchronize()
    assert torch.equal(o1, o2) and torch.equal(s1, s2[:126]) and torch.equal(s2[126], g.state[0])


@pytest.mark.parametrize("nseq", [63, 64, 65, 125, 126, 127])
def test_prefill_planning_limits(dev, nseq):
    """One and two planned sequences per lane, and the plan kernel above 126: empty and short
    sequences, chunk edges, tokens before the first and after the last, both cu_seqlens types."""
    lens = [(0, 1, 64, 65, 130, 20)[i % 6] for i in range(nseq)]
    inp = prefill_inputs(lens, hqk=2, hv=4, seed=nseq, with_state=True, gates="mild",
                         cu_dtype=torch.int64 if nseq % 2 else torch.int32, pad_tokens=7)
    inp.cu_seqlens += 3  # three tokens before the first sequence
    inp.cu_seqlens[-1] -= 3 if lens[-1] >= 3 else 0
    _run(dev, inp, f"planning limit N={nseq}")


@pytest.mark.parametrize("nseq", [3, 64, 300])
def test_prefill_gap_before_first_sequence(dev, nseq):
    """cu_seqlens[0] > 0: the leading tokens belong to no sequence and read as zero."""
    g = torch.Generator().manual_seed(7 + nseq)
    lens = [int(x) for x in torch.randint(1, 70, (nseq,), generator=g)]
    inp = prefill_inputs(lens, hqk=4, hv=8, seed=31, with_state=True, pad_tokens=53)
    inp.cu_seqlens = inp.cu_seqlens + 37  # 37 leading and 16 trailing gap tokens
    _run(dev, inp, f"lead gap N={nseq}")


@pytest.mark.parametrize("gates", ["strong", "mild", "none"])
def test_prefill_segments_long_memory(dev, gates):
    """Few (sequence, v-head) pairs: each long sequence is scanned as parallel segments
    whose states are chained (S_in M + R). Mild or no decay makes every segment's state
    carry into the next one."""
    _run(dev, prefill_inputs([2048], seed=41, with_state=True, gates=gates, state_std=0.1),
         f"segments gates={gates}")


@pytest.mark.parametrize("lens,hqk,hv,cut", [([3000, 300], 16, 32, True), ([3000], 4, 8, True),
                                             ([900, 0, 1400, 65], 4, 8, True),
                                             ([1500, 300], 16, 32, False)])
def test_prefill_segments_mixed(dev, lens, hqk, hv, cut):
    """Segmented and whole sequences in one call (short ones are not split), up to nine
    segments per sequence, empty sequences; and a mix that runs whole."""
    inp = prefill_inputs(lens, hqk=hqk, hv=hv, seed=43, with_state=True, gates="mild",
                         state_std=0.05)
    header = _run_with_header(dev, inp, f"segments lens={lens}")
    # a cut sequence: 3 jobs in pass A, 2 in pass C
    assert header[1] >= 3 and header[2] >= 2 if cut else header[1] == 0


@pytest.mark.parametrize("lens,hqk,hv,plan", [
    ([4096, 700, 650], 4, 8, (9, 7)),           # 64 chunks in 6 segments; 11-chunk ones whole in C
    ([3000, 200, 150, 100], 4, 8, (10, 4)),     # 47 chunks in 5 segments; the short ones whole in A
    # offered segments, none taken: equal lengths run whole in pass C, 4 and 10 jobs
    ([650, 640, 600, 655], 4, 8, (0, 4)),
    ([720, 700, 705, 690, 680, 660, 650, 640, 600, 710], 4, 8, (0, 10)),
    ([2500, 2400], 16, 32, (0, 2)),
    # a long prompt beside short ones
    ([1980, 20], 4, 8, (12, 6)),
    ([2400, 20, 20, 20], 4, 8, (10, 4)),
    ([6000, 100, 100, 100, 100, 100], 4, 8, (10, 3)),
    ([4000] + [20] * 11, 2, 4, (16, 3)),
    # all cut: 7 segment jobs each in pass A (224 pairs), 16 resumed segments in pass C
    ([8000, 7800, 7700, 7900], 4, 8, (28, 16)),
    ([8000, 0, 7800], 8, 16, (11, 6)),
    # ten of 44-50 chunks: cut in 3 both passes would need 8 waves and lose
    ([3000, 2900, 3100, 2950, 3050, 2800, 3200, 2850, 3150, 2990], 4, 8, (0, 10)),
    (varlen_lengths(8, seed=7), 4, 8, (0, 0)),  # 3-12 chunks: not offered
    # one sequence at 48 v-heads: whole, and in 4 segments where the call outgrows the cache
    ([4096], 24, 48, (0, 0)),
    ([8192], 24, 48, (5, 3)),
])
def test_prefill_segment_planner(dev, lens, hqk, hv, plan):
    """Segment plans on few sequences (mild decay, so every chained state carries into the next
    segment). Sequences of similar length all run whole in pass C with pass A empty; a long
    sequence is cut into segments while the short ones run whole in pass C beside its resumed
    segments, or in pass A beside its segment 0 and state maps. The one kernel of both passes
    then runs every body it holds (whole sequence, segment with outputs, both state maps) at
    every width (column split up to 64 (job, v-head) pairs, 4 waves up to 128, 8 above). The job
    counts the planner wrote (workspace header, cleared before: pass A, pass C) name the plan;
    a call that is not offered segments leaves both zero."""
    inp = prefill_inputs(lens, hqk=hqk, hv=hv, seed=59, with_state=True, gates="mild",
                         state_std=0.05)
    header = _run_with_header(dev, inp, f"planner {lens[:3]} x {hv}")
    assert (header[1], header[2]) == plan


@pytest.mark.parametrize("n,seed,use4", [(20, 4, True), (32, 6, False)])
def test_prefill_whole_scan_choice(dev, n, seed, use4):
    """Whole sequences with 129 to 256 (sequence, v-head) pairs: the prep kernel has them scanned
    by 4 waves when neither the mean load per CU nor the two jobs that meet on the CU filled last
    exceed 1.25 times the longest sequence (20 qk4_v8 sequences), else by 8 (32 sequences). The
    workspace header holds the counts (4-wave, 8-wave); the results hold the oracle bar."""
    inp = prefill_inputs(varlen_lengths(n, seed=seed), hqk=4, hv=8, seed=seed, with_state=True)
    header = _run_with_header(dev, inp, f"whole scan choice N={n}")
    assert (header[4], header[5]) == ((n, 0) if use4 else (0, n))


@pytest.mark.parametrize("seed,plan", [(0, "cut"), (1, "cut"), (2, "none"), (3, "whole"),
                                       (4, "cut"), (5, "cut"), (8, "cut"), (12, "whole"),
                                       (14, "cut")])
def test_prefill_segment_planner_random(dev, seed, plan):
    """Random mixes in the segment regime (2 to 10 sequences, qk4_v8 heads, N HV 3 <= 256):
    long sequences that may be cut beside short and empty ones, so plans mix cut sequences,
    whole jobs in either pass and the all-whole plan; mild decay keeps every chained state
    significant. The job counts say which kind of plan each mix took ("none": too short to be
    offered segments)."""
    rng = np.random.default_rng(1000 + seed)
    n = int(rng.integers(2, 11))
    lens = [int(rng.choice([rng.integers(0, 3), rng.integers(1, 400), rng.integers(400, 1400),
                             rng.integers(1400, 3200)], p=[0.1, 0.35, 0.35, 0.2]))
            for _ in range(n)]
    header = _run_with_header(dev, prefill_inputs(lens, hqk=4, hv=8, seed=70 + seed, with_state=True,
                                                  gates="mild", state_std=0.05),
                              f"planner mix {seed} lens={lens}")
    jobs = header[1:3]
    if plan == "cut":
        assert jobs[0] >= 3 and jobs[1] >= 2
    else:
        assert jobs == ([0, n] if plan == "whole" else [0, 0])


@pytest.mark.parametrize("short", [68, 128])
def test_prefill_long_sequences_among_many_plan_kernel(dev, short):
    """Two long sequences among 68 or 128 short ones with one v-head: every sequence is scanned
    whole (the job planner, and with it segments, serves up to 64 sequences), and above 126
    sequences the plan kernel builds the tables."""
    rng = np.random.default_rng(77)
    lens = [int(x) for x in rng.integers(0, 40, short)] + [2500, 1900]
    _run(dev, prefill_inputs(lens, hqk=1, hv=1, seed=78, with_state=True, gates="mild",
                             state_std=0.05), f"plan-kernel segments N={len(lens)}")


@pytest.mark.parametrize("lens,hqk,hv,cut", [([2048], 16, 32, True), ([3000, 20], 16, 32, True),
                                             ([2048, 1100], 4, 8, True),
                                             ([1400, 0, 1200, 900], 4, 8, True),
                                             ([2048, 1100], 16, 32, False)])
def test_prefill_segments_inplace_state(dev, lens, hqk, hv, cut):
    """Segmented scan with new_state aliasing state: pass A reads the initial state only in
    segment 0's job, and only the last segment's pass-C job writes the final state; whole
    sequences read and write theirs in one job of either pass."""
    inp = prefill_inputs(lens, hqk=hqk, hv=hv, seed=53, with_state=True, gates="mild",
                         state_std=0.05)
    header = _run_with_header(dev, inp, f"segments in-place {lens}", inplace=True)
    assert header[1] >= 3 and header[2] >= 2 if cut else header[1] == 0


def test_prefill_segments_match_whole_sequence_scan(dev):
    """The segmented scan and the whole-sequence scan (tuning variant 2) agree."""
    from gdn_hip.api import set_prefill_variant
    inp = prefill_inputs([1800], seed=47, with_state=True, gates="mild").to(dev)
    out_s, ns_s = gdn_prefill(*inp.args())
    try:
        set_prefill_variant(2)
        out_w, ns_w = gdn_prefill(*inp.args())
    finally:
        set_prefill_variant(0)
    torch.cuda.synchronize()
    vo = check_output(out_s, out_w.float())
    vs = check_state(ns_s, ns_w)
    print(f"[segmented vs whole] output {vo} | state {vs}", flush=True)
    assert vo.ok and vs.ok


@pytest.mark.parametrize("lens", [[300, 77, 1000], [2048]])
def test_prefill_extreme_gates(dev, lens):
    """Extreme gate inputs (softplus x > 20 branch, beta ~ 0 / ~ 1, alpha exactly 1 / 0)
    through whole-sequence and segmented scans."""
    inp = with_extreme_gates(prefill_inputs(lens, seed=63, with_state=True), seed=64)
    _run(dev, inp, f"extreme gates lens={lens}")


def _random_case(i):
    """Seeded random prefill case: sequence count and lengths (empty, sub-chunk, chunk
    multiples, long), head layout, gate regime, initial state, padding tokens, cu dtype."""
    rng = np.random.default_rng(7100 + i)
    hqk, hv = [(16, 32), (4, 8), (8, 16), (2, 8)][i % 4]
    n = int(rng.choice([1, 1, 2, 3, 4, 7, 12, 25]))
    kind = rng.choice(["empty", "short", "chunk", "medium", "long"], size=n,
                      p=[0.1, 0.2, 0.1, 0.3, 0.3])
    lens = [int({"empty": 0, "short": rng.integers(1, 64), "chunk": 64 * rng.integers(1, 6),
                 "medium": rng.integers(65, 800), "long": rng.integers(800, 3200)}[k])
            for k in kind]
    while sum(lens) > 5000:
        lens = [x // 2 for x in lens]
    gates = str(rng.choice(["strong", "mild", "none", "extreme"]))
    inp = prefill_inputs(lens, hqk=hqk, hv=hv, seed=7200 + i,
                         with_state=bool(rng.integers(0, 4) > 0),
                         gates="strong" if gates == "extreme" else gates, state_std=0.05,
                         cu_dtype=torch.int64 if rng.integers(0, 2) else torch.int32,
                         pad_tokens=int(rng.choice([0, 0, 3, 70])))
    if gates == "extreme":
        inp = with_extreme_gates(inp, seed=7300 + i)
    return inp, f"random {i}: hqk={hqk} hv={hv} gates={gates} lens={lens}"


@pytest.mark.parametrize("i", range(10))
def test_prefill_random_cases(dev, i):
    """Seeded random mixes of 1 to 25 sequences (short and empty ones next to long ones, whole
    and in segments) under every gate regime."""
    inp, label = _random_case(i)
    _run(dev, inp, label)


def test_prefill_long_sequence_64k(dev):
    """One 65536-token sequence (1024 chunks): sixteen segments of ~64 chunks with their state
    chain, mild decay so every segment's state carries into the next."""
    inp = prefill_inputs([65536], hqk=1, hv=2, seed=97, with_state=True, gates="mild",
                         state_std=0.05)
    _run(dev, inp, "1 x 65536, hqk=1 hv=2")


def test_prefill_and_decode_on_concurrent_streams(dev):
    """Two prefills in flight at once on two streams (each stream has its own cached
    workspace) and a decode on a third; every result matches the oracle."""
    from gdn_hip.inputs import decode_inputs
    ia = prefill_inputs([700, 300, 45], seed=201, with_state=True)
    ib = prefill_inputs([1500], seed=202, with_state=True, gates="mild", state_std=0.05)
    idc = decode_inputs(8, seed=203)
    ref_a, ref_b = _oracle(ia), _oracle(ib)
    ref_d = O.decode(*idc.args())
    ga, gb, gd = ia.to(dev), ib.to(dev), idc.to(dev)
    torch.cuda.synchronize()
    s1, s2, s3 = torch.cuda.Stream(dev), torch.cuda.Stream(dev), torch.cuda.Stream(dev)
    with torch.cuda.stream(s1):
        oa, na = gdn_prefill(*ga.args())
    with torch.cuda.stream(s2):
        ob, nb = gdn_prefill(*gb.args())
    with torch.cuda.stream(s3):
        od, nd = gdn_decode(*gd.args())
    torch.cuda.synchronize()
    _check(oa, na, *ref_a, "stream 1 prefill")
    _check(ob, nb, *ref_b, "stream 2 prefill")
    _check(od, nd, *ref_d, "stream 3 decode")


def test_prefill_in_graph(dev):
    """gdn_prefill captured in a HIP graph (plan, prep and scan launches): every replay, with
    eager work and a sync between replays, reproduces the eager call bit for bit."""
    inp = prefill_inputs([500, 64, 1300, 7], seed=311, with_state=True)
    ref_out, ref_ns = _oracle(inp)
    g = inp.to(dev)
    T, N = g.q.shape[0], len(inp.seqlens)
    out = torch.empty((T, 32, 128), dtype=torch.bfloat16, device=dev)
    ns = torch.empty((N, 32, 128, 128), dtype=torch.float32, device=dev)
    gdn_prefill(*g.args(), output=out, new_state=ns)
    torch.cuda.synchronize()
    _check(out, ns, ref_out, ref_ns, "eager")
    eager_out, eager_ns = out.clone(), ns.clone()
    side = torch.cuda.Stream(dev)
    side.wait_stream(torch.cuda.current_stream(dev))
    with torch.cuda.stream(side):
        gdn_prefill(*g.args(), output=out, new_state=ns)
    torch.cuda.current_stream(dev).wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        gdn_prefill(*g.args(), output=out, new_state=ns)
    for r in range(3):
        out.zero_()
        ns.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager_out), f"replay {r}: output differs"
        assert torch.equal(ns, eager_ns), f"replay {r}: new_state differs"


@pytest.mark.parametrize("lens,hqk,hv", [
    ([1900] + [1 + (37 * i) % 130 for i in range(95)], 4, 8),  # queued 8-wave scan <-> wide
    ([2400, 20, 20, 20], 4, 8),                                # segments <-> whole sequences
    ([1500, 400] + [100] * 18, 4, 8),                          # 4 waves <-> 8 waves
])
def test_prefill_graph_replays_other_lengths(dev, lens, hqk, hv):
    """A captured prefill replayed with the lengths of its sequences changed in cu_seqlens: the
    planner chooses anew on every replay (its job counts and queues start from zero each time),
    and each equals the eager call on the same lengths bit for bit."""
    n, T = len(lens), sum(lens)
    g = prefill_inputs(lens, hqk=hqk, hv=hv, seed=7, with_state=True, gates="mild").to(dev)
    skewed = g.cu_seqlens.clone()
    even = torch.tensor([T * i // n for i in range(n + 1)], dtype=torch.int32, device=dev)
    eager = []
    for cu in (skewed, even):
        g.cu_seqlens.copy_(cu)
        eager.append(gdn_prefill(*g.args()))
    assert not torch.equal(eager[0][0], eager[1][0])
    out, ns = torch.empty_like(eager[0][0]), torch.empty_like(eager[0][1])
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        gdn_prefill(*g.args(), output=out, new_state=ns)
    for r in range(5):
        i = (0, 1, 1, 0, 0)[r]
        g.cu_seqlens.copy_((skewed, even)[i])
        out.zero_()
        ns.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager[i][0]), f"replay {r}: output differs"
        assert torch.equal(ns, eager[i][1]), f"replay {r}: new_state differs"


def test_prefill_graphs_keep_their_own_workspaces(dev):
    """Two graphs captured one after the other, the second needing a larger workspace, and
    an eager call in between: each graph keeps its own workspace, so replaying the first
    after the second (and after eager work) still reproduces its eager result bit for bit."""
    def setup(lens, seed):
        g = prefill_inputs(lens, seed=seed, with_state=True).to(dev)
        T, N = g.q.shape[0], len(lens)
        out = torch.empty((T, 32, 128), dtype=torch.bfloat16, device=dev)
        ns = torch.empty((N, 32, 128, 128), dtype=torch.float32, device=dev)
        gdn_prefill(*g.args(), output=out, new_state=ns)
        torch.cuda.synchronize()
        return g, out, ns, out.clone(), ns.clone()

    ga, oa, na, ea_o, ea_n = setup([130, 70], 401)
    gb, ob, nb, eb_o, eb_n = setup([900, 1100, 640], 402)
    graphs = []
    for g, o, n in ((ga, oa, na), (gb, ob, nb)):
        side = torch.cuda.Stream(dev)  # warm-up on a side stream, as torch.cuda.graph asks
        side.wait_stream(torch.cuda.current_stream(dev))
        with torch.cuda.stream(side):
            gdn_prefill(*g.args(), output=o, new_state=n)
        torch.cuda.current_stream(dev).wait_stream(side)
        torch.cuda.synchronize()
        gr = torch.cuda.CUDAGraph()
        with torch.cuda.graph(gr):
            gdn_prefill(*g.args(), output=o, new_state=n)
        graphs.append(gr)
    gdn_prefill(*gb.args())  # eager work between the replays
    for r, (gr, o, n, eo, en) in enumerate([(graphs[0], oa, na, ea_o, ea_n),
                                            (graphs[1], ob, nb, eb_o, eb_n),
                                            (graphs[0], oa, na, ea_o, ea_n)]):
        o.zero_()
        n.zero_()
        torch.cuda.synchronize()
        gr.replay()
        torch.cuda.synchronize()
        print(f"[two graphs] replay {r} bitwise: {torch.equal(o, eo)} {torch.equal(n, en)}",
              flush=True)
        assert torch.equal(o, eo) and torch.equal(n, en), f"replay {r} differs"


def test_prefill_graph_workspaces_released_with_the_graphs(dev):
    """A captured prefill holds a workspace of its own until the caller, having destroyed the
    graph, calls release_workspace(graphs=True); the graph's replay before that matches its
    eager result, and a new capture after the release works again."""
    from gdn_hip import graph_workspace_bytes

    g = prefill_inputs([300, 41], seed=77, with_state=True).to(dev)
    T, N = g.q.shape[0], 2
    out = torch.empty((T, 32, 128), dtype=torch.bfloat16, device=dev)
    ns = torch.empty((N, 32, 128, 128), dtype=torch.float32, device=dev)
    gdn_prefill(*g.args(), output=out, new_state=ns)
    torch.cuda.synchronize()
    eo, en = out.clone(), ns.clone()
    need = _lib.load().gdn_prefill_workspace_size(T, N, 16, 32, 128)
    for rnd in range(2):
        before = graph_workspace_bytes()
        gr = torch.cuda.CUDAGraph()
        with torch.cuda.graph(gr):
            gdn_prefill(*g.args(), output=out, new_state=ns)
        assert graph_workspace_bytes() - before >= need
        out.zero_()
        ns.zero_()
        torch.cuda.synchronize()
        gr.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eo) and torch.equal(ns, en), f"round {rnd}: replay differs"
        del gr
        torch.cuda.synchronize()
        release_workspace(graphs=True)
        assert graph_workspace_bytes() == 0


def test_prefill_fast_path_taken_and_exact(dev):
    """A destination-passing prefill outside capture goes through the C++ fast path: it
    launches (returns 0), matches the oracle and equals the Python path bit for bit; after
    release_workspace() it allocates a fresh workspace and still matches."""
    from gdn_hip import _lib
    from gdn_hip.api import release_workspace

    fast = _lib.fast()
    assert fast is not None
    inp = prefill_inputs([300, 64, 129, 1], hqk=4, hv=8, seed=88, with_state=True)
    ref_o, ref_s = _oracle(inp)
    g = inp.to(dev)
    T, N = g.q.shape[0], len(inp.seqlens)
    out = torch.empty((T, 8, 128), dtype=torch.bfloat16, device=dev)
    ns = torch.empty((N, 8, 128, 128), dtype=torch.float32, device=dev)
    assert fast.prefill(*g.args(), out, ns, 0) == 0
    torch.cuda.synchronize()
    _check(out, ns, ref_o, ref_s, "prefill fast path")
    import ctypes

    from gdn_hip.api import _prefill_marshal
    o2, n2 = torch.empty_like(out), torch.empty_like(ns)
    P, _, _, copy_back, keep, stream = _prefill_marshal(*g.args(), o2, n2)
    assert not copy_back
    _lib.check(_lib.load().gdn_prefill_launch(ctypes.byref(P), ctypes.c_void_p(
        stream.cuda_stream)), "gdn_prefill_launch")
    torch.cuda.synchronize()
    assert torch.equal(out, o2) and torch.equal(ns, n2)
    release_workspace()
    o3, n3 = gdn_prefill(*g.args(), torch.empty_like(out), torch.empty_like(ns))
    torch.cuda.synchronize()
    assert torch.equal(out, o3) and torch.equal(ns, n3)


def test_prefill_fast_path_allocates_missing_outputs(dev):
    """A prefill without output and new_state: allocated by the fast path, equal to the
    destination-passing call; empty inputs still go to the general path."""
    fast = _lib.fast()
    g = prefill_inputs([70, 130], hqk=4, hv=8, seed=90, with_state=True).to(dev)
    eo = torch.empty((200, 8, 128), dtype=torch.bfloat16, device=dev)
    en = torch.empty_like(g.state)
    assert fast.prefill(*g.args(), eo, en, 0) == 0
    r = fast.prefill_alloc(*g.args(), None, None, 0)
    assert r is not None
    o2, n2 = gdn_prefill(*g.args(), output=eo.clone())
    torch.cuda.synchronize()
    for o, n in (r, (o2, n2)):
        assert torch.equal(o, eo) and torch.equal(n, en)
    e = prefill_inputs([0, 0], seed=2, with_state=True).to(dev)
    assert fast.prefill_alloc(*e.args(), None, None, 0) is None
    o, n = gdn_prefill(*e.args())
    assert o.shape[0] == 0 and torch.equal(n, e.state)


def test_prefill_fast_path_declines_capture_and_odd_layouts(dev):
    """Graph capture, a strided output and empty inputs go to the general path."""
    from gdn_hip import _lib

    fast = _lib.fast()
    g = prefill_inputs([70, 30], seed=89, with_state=True).to(dev)
    T = g.q.shape[0]
    out = torch.empty((T, 32, 128), dtype=torch.bfloat16, device=dev)
    ns = torch.empty((2, 32, 128, 128), dtype=torch.float32, device=dev)
    wide = torch.empty((T, 32, 256), dtype=torch.bfloat16, device=dev)
    assert fast.prefill(*g.args(), wide[..., ::2], ns, 0) == 1
    e = prefill_inputs([0, 0], seed=2, with_state=True).to(dev)
    assert fast.prefill(*e.args(), torch.empty((0, 32, 128), dtype=torch.bfloat16, device=dev),
                        torch.empty_like(e.state), 0) == 1
    fast.prefill(*g.args(), out, ns, 0)  # warm the stream's cached workspace
    torch.cuda.synchronize()
    side = torch.cuda.Stream(dev)
    side.wait_stream(torch.cuda.current_stream(dev))
    with torch.cuda.stream(side):
        gdn_prefill(*g.args(), output=out, new_state=ns)
    torch.cuda.current_stream(dev).wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        rc = fast.prefill(*g.args(), out, ns, 0)
    assert rc == 1
