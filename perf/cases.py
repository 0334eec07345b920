"""Performance cases of the Gated Delta Net decode step and prefill.

Each listed case is one call (or one replay of a model's captured layers) as
a serving program makes it, through the package's public entry points:

* ``kernel_hip``: one decode step in place on the layer's running state;
* ``run``: the value-returning decode step;
* ``DecodeLayers.replay``: the decode steps of a model's GDN layers;
* ``kernel_prefill_hip``: a prefill into preallocated buffers;
* ``prefill_run``: the value-returning prefill.

Inputs follow the model: q and k ~ N(0, 1), with unit rows where the call
does not normalise them itself (``l2``); v, a, b ~ N(0, 1); states ~
N(0, 0.05^2); A_log = log U[1, 16]; dt_bias ~ U[-1, 1].  K = V = 128.
"""

from __future__ import annotations

import math

import torch

import flashinfer_competition_codebase_amd as gdn
from flashinfer_competition_codebase_amd.serving import DecodeLayers

DIM = 128
L2_EPS = 1e-6
SOFTPLUS_THRESHOLD = 20.0


def _decode(name, entry, B, H, HV, T=1, state="fp32", l2=True):
    return dict(name=name, kind="decode", entry=entry, B=B, T=T, H=H, HV=HV, state=state, l2=l2)


def _prefill(name, entry, lens, H, HV, state="fp32", l2=True):
    return dict(name=name, kind="prefill", entry=entry, lens=lens, H=H, HV=HV, state=state, l2=l2)


def listed():
    return [
        # one user's decode step on a tensor-parallel shard: launch latency
        _decode("decode_b1_qk4v8", "dps", 1, 4, 8, l2=False),
        # an odd-sized continuous batch on that shard
        _decode("decode_b37_qk4v8", "dps", 37, 4, 8, l2=False),
        # a large serving batch with the whole model's heads (the benchmark's headline)
        _decode("decode_b256_qk16v32", "dps", 256, 16, 32),
        # speculative decoding: four draft tokens verified per step, bf16 state
        _decode("decode_b64_t4_bf16", "dps", 64, 16, 32, T=4, state="bf16"),
        # two tokens per step through the value-returning form, an odd batch
        _decode("decode_b101_t2_run", "run", 101, 8, 32, T=2),
        # one user's decode step through a model's 48 GDN layers, captured once
        dict(name="decode_layers48_b1", kind="layers", layers=48, B=1, H=16, HV=32, l2=True),
        # the shortest prompt: a few tokens continuing a sequence
        _prefill("prefill_1x6_qk4v8", "dps", "6", 4, 8, l2=False),
        # a few short prompts of different lengths, from nothing
        _prefill("prefill_ragged4_qk4v8", "run", "100,217,300,383", 4, 8, state="none", l2=False),
        # a batch of medium prompts continuing their sequences, on a shard
        _prefill("prefill_16x1024_qk4v8", "dps", "16*1024", 4, 8, l2=False),
        # one long document on a shard
        _prefill("prefill_1x16384_qk4v8", "dps", "16384", 4, 8, l2=False),
        # a large batch of prompts with the whole model's heads
        _prefill("prefill_64x512_qk16v32", "dps", "64*512", 16, 32),
        # a ragged batch of new prompts with the whole model's heads
        _prefill("prefill_ragged12_qk16v32", "dps",
                 "1873,64,911,2048,333,1500,7,1201,640,129,1777,450", 16, 32, state="none"),
    ]


def _lens(case):
    """Sequence lengths: "64*512" or "100,217", items in order."""
    lens = []
    for item in case["lens"].split(","):
        n, _, length = item.rpartition("*")
        lens += [int(length)] * (int(n) if n else 1)
    return lens


def _log_int(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


# (q/k heads, v-heads): the shard's and the whole model's, and other GVA ratios
HEADS = [(4, 8), (16, 32), (8, 32), (8, 16), (2, 4), (3, 12)]


def draw(rng):
    """One case of the same ranges: decode batches of 1 to 8192 heads, 1 to 4
    tokens; prefills of 1 to 16384 tokens a sequence, up to 32768 tokens."""
    H, HV = rng.choice(HEADS)
    l2 = rng.random() < 0.6
    u = rng.random()
    if u < 0.10:
        return dict(kind="layers", layers=rng.randint(8, 48), B=rng.randint(1, 4), H=H, HV=HV,
                    l2=l2)
    if u < 0.50:
        T = rng.choice([1, 1, 1, 2, 3, 4])
        state = "bf16" if rng.random() < 0.3 else "fp32"
        entry = "run" if rng.random() < 0.2 else "dps"
        B = _log_int(rng, 1, min(512, 8192 // HV))
        return dict(kind="decode", entry=entry, B=B, T=T, H=H, HV=HV, state=state, l2=l2)
    entry = "run" if rng.random() < 0.25 else "dps"
    state = "none" if rng.random() < 0.4 else "fp32"
    # token x v-head products up to the largest listed batch's
    total = _log_int(rng, 1, 32768 if HV >= 16 else 49152)
    most = max(1, min(64, 2048 // HV, total))
    N = 1 if rng.random() < 0.3 else _log_int(rng, 1, most)
    N = max(N, -(-total // 16384))
    if rng.random() < 0.4:
        lens = f"{N}*{max(1, total // N)}"
    else:                                          # ragged: lengths over a factor of ~20
        w = [math.exp(rng.uniform(-3.0, 0.0)) for _ in range(N)]
        s = sum(w)
        lens = ",".join(str(min(16384, max(1, int(total * x / s)))) for x in w)
    return dict(kind="prefill", entry=entry, lens=lens, H=H, HV=HV, state=state, l2=l2)


def _inputs(case, seed):
    """q, k, v, state, A_log, a, dt_bias, b with the token axes of the entry,
    made on the GPU from the seed."""
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(seed)
    H, HV = case["H"], case["HV"]
    if case["kind"] == "prefill":
        lens = _lens(case)
        lead, n_seq = (sum(lens),), (len(lens),)
    elif case["kind"] == "layers":
        lead, n_seq = (case["layers"], case["B"], 1), (case["layers"], case["B"])
    else:
        lead, n_seq = (case["B"], case["T"]), (case["B"],)

    def rand(*shape):
        return torch.randn(*shape, generator=g, device=dev)

    def rows(*shape):
        x = rand(*shape)
        if not case["l2"]:
            x = x / x.norm(dim=-1, keepdim=True).clamp_min(1e-6)
        return x.to(torch.bfloat16)

    per_head = (case["layers"], HV) if case["kind"] == "layers" else (HV,)
    t = dict(
        q=rows(*lead, H, DIM),
        k=rows(*lead, H, DIM),
        v=rand(*lead, HV, DIM).to(torch.bfloat16),
        state=None,
        A_log=torch.log(torch.rand(*per_head, generator=g, device=dev) * 15.0 + 1.0),
        a=rand(*lead, HV).to(torch.bfloat16),
        dt_bias=torch.rand(*per_head, generator=g, device=dev) * 2.0 - 1.0,
        b=rand(*lead, HV).to(torch.bfloat16),
        scale=1.0 / math.sqrt(DIM),
    )
    kind = case.get("state", "fp32")
    if kind != "none":
        t["state"] = rand(*n_seq, HV, DIM, DIM).mul_(0.05)
        if kind == "bf16":
            t["state"] = t["state"].to(torch.bfloat16)
    return t


def _cu_seqlens(case):
    cu = [0]
    for n in _lens(case):
        cu.append(cu[-1] + n)
    return torch.tensor(cu, dtype=torch.int32, device="cuda")


def prepare(case, seed):
    t = _inputs(case, seed)
    l2 = case["l2"]
    if case["kind"] == "layers":
        output = torch.empty_like(t["v"])
        layers = DecodeLayers(
            [dict(q=t["q"][i], k=t["k"][i], v=t["v"][i], state=t["state"][i],
                  A_log=t["A_log"][i], a=t["a"][i], dt_bias=t["dt_bias"][i], b=t["b"][i],
                  scale=t["scale"], output=output[i], new_state=t["state"][i])
             for i in range(case["layers"])], use_qk_l2norm=l2)
        layers.capture()
        return dict(call="layers", layers=layers, output=output, state=t["state"], tensors=t)
    if case["kind"] == "decode":
        if case["entry"] == "dps":                 # in place on the running state
            t["output"] = torch.empty_like(t["v"])
            t["new_state"] = t["state"]
        return dict(call="decode", entry=case["entry"], args=t, l2=l2)
    t["cu_seqlens"] = _cu_seqlens(case)
    if case["entry"] == "dps":
        n_seq = t["cu_seqlens"].numel() - 1
        t["output"] = torch.empty_like(t["v"])
        t["new_state"] = torch.empty(n_seq, case["HV"], DIM, DIM, device="cuda")
    return dict(call="prefill", entry=case["entry"], args=t, l2=l2)


def run(state):
    if state["call"] == "layers":
        state["layers"].replay()
        return state["output"], state["state"]
    t, l2 = state["args"], state["l2"]
    if state["call"] == "decode":
        if state["entry"] == "run":
            return gdn.run(**t, use_qk_l2norm=l2)
        gdn.kernel_hip(**t, use_qk_l2norm=l2)
        return t["output"], t["new_state"]
    if state["entry"] == "run":
        return gdn.prefill_run(**t, use_qk_l2norm=l2)
    gdn.kernel_prefill_hip(**t, use_qk_l2norm=l2)
    return t["output"], t["new_state"]


def _token_counts(case):
    """(tokens in all, sequences in all, states read, bytes of a state element)."""
    if case["kind"] == "prefill":
        lens = _lens(case)
        return sum(lens), len(lens), 0 if case["state"] == "none" else len(lens), 4
    if case["kind"] == "layers":
        n = case["layers"] * case["B"]
        return n, n, n, 4
    return (case["B"] * case["T"], case["B"], case["B"], 2 if case["state"] == "bf16" else 4)


def work(case):
    """q, k, v, a, b and the states read once, the outputs and states written
    once; per token and v-head the recurrence's decay (1), two dot products
    and rank-one update (2 each) per state element."""
    tokens, seqs, states_in, elem = _token_counts(case)
    H, HV = case["H"], case["HV"]
    per_token = 2 * (2 * H * DIM + 2 * HV * DIM + 2 * HV)
    state_bytes = HV * DIM * DIM * elem
    return {"bytes": tokens * per_token + (states_in + seqs) * state_bytes + 8 * HV,
            "flops": tokens * HV * 7 * DIM * DIM}


def tolerance(case):
    # bf16 outputs (half an ulp each side, ~1.7e-3 of the 64-bit result) set
    # the bar; a result near a rounding boundary may land one ulp (2^-8) away.
    return {"rel": 6e-3, "max": 2e-2}


def _exact_steps(q, k, v, S, logg, beta, scale, l2, lens):
    """The recurrence in 64 bits, token after token over all sequences at
    once: q, k [N, T, HV, K], v [N, T, HV, V], S [N, HV, V, K], sequences in
    order of falling length (lens).  Returns (output [N, T, HV, V], S)."""
    if l2:
        q = q * torch.rsqrt((q * q).sum(-1, keepdim=True) + L2_EPS)
        k = k * torch.rsqrt((k * k).sum(-1, keepdim=True) + L2_EPS)
    out = torch.zeros_like(v)
    g = torch.exp(logg)
    n = len(lens)
    for t in range(lens[0]):
        while lens[n - 1] <= t:
            n -= 1
        Sn = S[:n]
        Sn.mul_(g[:n, t, :, None, None])
        kt = k[:n, t, :, :, None].contiguous()
        d = beta[:n, t, :, None] * (v[:n, t] - torch.matmul(Sn, kt).squeeze(-1))
        Sn.add_(d[..., :, None] * kt.transpose(-1, -2))
        out[:n, t] = scale * torch.matmul(Sn, q[:n, t, :, :, None].contiguous()).squeeze(-1)
    return out, S


@torch.no_grad()
def exact(case, seed):
    t = _inputs(case, seed)
    f64 = torch.float64
    H, HV = case["H"], case["HV"]
    shape = t["v"].shape
    if case["kind"] == "layers":                   # independent layers: more sequences
        lens = [1] * (case["layers"] * case["B"])
    elif case["kind"] == "decode":
        lens = [case["T"]] * case["B"]
    else:
        lens = _lens(case)
    n, most = len(lens), max(lens)
    order = sorted(range(n), key=lambda i: -lens[i])
    # token rows of the packed inputs, [n, most] in falling length order
    first, at = [], 0
    for length in lens:
        first.append(at)
        at += length
    rows = torch.tensor([[first[i] + min(s, lens[i] - 1) for s in range(most)] for i in order],
                        device="cuda")
    keep = torch.tensor([[s < lens[i] for s in range(most)] for i in order], device="cuda")

    def tokens(x, heads, width):
        return x.reshape(-1, heads, width)[rows].to(f64)

    q = tokens(t["q"], H, DIM).repeat_interleave(HV // H, dim=2)
    k = tokens(t["k"], H, DIM).repeat_interleave(HV // H, dim=2)
    v = tokens(t["v"], HV, DIM)
    per_head = [t[x].to(f64) for x in ("A_log", "dt_bias")]
    if case["kind"] == "layers":
        per_head = [x.repeat_interleave(case["B"], dim=0)[:, None, :] for x in per_head]
    A_log, dt_bias = per_head
    x = t["a"].reshape(-1, HV)[rows].to(f64) + dt_bias
    sp = torch.where(x > SOFTPLUS_THRESHOLD, x, torch.log1p(torch.exp(x)))
    logg = -torch.exp(A_log) * sp
    beta = torch.sigmoid(t["b"].reshape(-1, HV)[rows].to(f64))
    if t["state"] is None:
        S = torch.zeros(n, HV, DIM, DIM, dtype=f64, device="cuda")
    else:
        S = t["state"].reshape(-1, HV, DIM, DIM)[torch.tensor(order, device="cuda")].to(f64)
    out, S = _exact_steps(q, k, v, S, logg, beta, t["scale"], case["l2"],
                          [lens[i] for i in order])
    output = torch.zeros(at, HV, DIM, dtype=f64, device="cuda")
    output[rows[keep]] = out[keep]
    new_state = torch.empty_like(S)
    new_state[torch.tensor(order, device="cuda")] = S
    lead = (case["layers"], case["B"]) if case["kind"] == "layers" else (n,)
    return output.reshape(shape), new_state.reshape(*lead, HV, DIM, DIM)
