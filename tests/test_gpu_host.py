"""The native call path (csrc/host.cpp) against the Python path it stands in
for: the calls it takes give the same bits, the calls it does not take reach
the Python path's conversions and errors (needs a HIP device)."""

from __future__ import annotations

import sys

import pytest
import torch

import flashinfer_competition_codebase_amd as gdn
from flashinfer_competition_codebase_amd import _lib
from flashinfer_competition_codebase_amd import kernel as kmod
from flashinfer_competition_codebase_amd import prefill as pmod
from oracle.gdn_decode_oracle import make_inputs
from oracle.gdn_prefill_oracle import make_prefill_inputs

pytestmark = pytest.mark.gpu


def _announce(case):
    sys.stdout.write(f"[gpu case] {case}\n")
    sys.stdout.flush()


@pytest.fixture(scope="module", autouse=True)
def _bound():
    _lib.bind_host()


def _dev(t, device):
    return {n: (x.to(device) if isinstance(x, torch.Tensor) else x) for n, x in t.items()}


def _host_prefill(t, l2=False, output=None, new_state=None):
    return _lib.bound_host.prefill(t["q"], t["k"], t["v"], t["state"], t["A_log"], t["a"],
                                   t["dt_bias"], t["b"], t["cu_seqlens"], t["scale"], output,
                                   new_state, l2)


PREFILLS = {
    "token path": ([6], 4, 8, True),
    "token path, several, no state": ([3, 1, 20], 3, 12, False),
    "one chunk": ([64], 4, 8, True),
    "two launches": ([65, 7], 4, 8, True),
    "offsets kernel": ([70] + [1] * 70, 4, 8, False),
    "segments": ([1024], 2, 4, True),
    "token path, many heads": ([56], 256, 256, True),
}


@pytest.mark.parametrize("case", list(PREFILLS))
@pytest.mark.parametrize("side_stream", [False, True])
def test_native_prefill_matches_the_python_path(case, side_stream, hip_device):
    lens, H, HV, with_state = PREFILLS[case]
    _announce(f"native prefill: {case}, side stream {side_stream}")
    t = _dev(make_prefill_inputs(lens, H, HV, seed=801, with_state=with_state), hip_device)
    stream = torch.cuda.Stream() if side_stream else torch.cuda.current_stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        args = (t["q"], t["k"], t["v"], t["state"], t["A_log"], t["a"], t["dt_bias"], t["b"],
                t["cu_seqlens"], t["scale"])
        ref_o, ref_s = pmod._prefill_run_checked(*args, False)
        code, out, st = _host_prefill(t)
        assert code == 0 and not out.requires_grad
        out2, st2 = torch.empty_like(out), torch.empty_like(st)
        assert _host_prefill(t, False, out2, st2) == 0
        assert torch.equal(out, ref_o) and torch.equal(st, ref_s)
        assert torch.equal(out2, ref_o) and torch.equal(st2, ref_s)
        if with_state:                              # in place
            t["state"] = t["state"].clone()
            assert _host_prefill(t, False, out2, t["state"]) == 0
            assert torch.equal(t["state"], ref_s)
    torch.cuda.current_stream().wait_stream(stream)


@pytest.mark.parametrize("B,T,H,HV,dtype,l2", [
    (1, 1, 4, 8, torch.float32, False), (3, 2, 3, 12, torch.float32, True),
    (5, 4, 2, 2, torch.bfloat16, True), (2, 1, 4, 8, None, False),
])
@pytest.mark.parametrize("flat_gates", [False, True])
def test_native_decode_matches_the_python_path(B, T, H, HV, dtype, l2, flat_gates, hip_device):
    _announce(f"native decode B={B} T={T} qk{H}_v{HV} {dtype} l2={l2} flat={flat_gates}")
    t = _dev(make_inputs(B, H, HV, seed=811, T=T), hip_device)
    t["state"] = None if dtype is None else t["state"].to(dtype)
    if flat_gates and T == 1:
        t["a"], t["b"] = t["a"].view(B, HV), t["b"].view(B, HV)
    names = ("q", "k", "v", "state", "A_log", "a", "dt_bias", "b", "scale")
    ref = kmod._run_checked(*[t[n] for n in names], l2)
    code, out, st = _lib.bound_host.decode_run(*[t[n] for n in names], l2)
    assert code == 0 and torch.equal(out, ref[0]) and torch.equal(st, ref[1])
    got = gdn.run(**t, use_qk_l2norm=l2)
    assert torch.equal(got[0], ref[0]) and torch.equal(got[1], ref[1])


def test_calls_the_native_path_leaves_to_python(hip_device):
    """Conversions (int64 cu_seqlens, tensor scales, integer flags) work as
    before; malformed calls raise what they raised."""
    _announce("native path: conversions and refusals")
    t = _dev(make_prefill_inputs([40, 90], 4, 8, seed=821), hip_device)
    ref_o, ref_s = gdn.prefill_run(**t)
    other = {
        "cu_seqlens": t["cu_seqlens"].long(),
        "scale": torch.tensor(t["scale"], device=hip_device),
    }
    for n, x in other.items():
        assert _host_prefill({**t, n: x}) is None
        o, s = gdn.prefill_run(**{**t, n: x})
        assert torch.equal(o, ref_o) and torch.equal(s, ref_s), n
    assert _host_prefill(t, 0) is None                       # a flag that is no bool
    o, s = gdn.prefill_run(**t, use_qk_l2norm=0)
    assert torch.equal(o, ref_o) and torch.equal(s, ref_s)
    bad = {
        "q": t["q"].float(), "k": t["k"][:-1], "v": t["v"].transpose(1, 2).contiguous(),
        "state": t["state"].transpose(2, 3), "A_log": t["A_log"].double(), "a": t["a"].cpu(),
        "dt_bias": t["dt_bias"][:-1], "b": None, "cu_seqlens": t["cu_seqlens"].float(),
    }
    for n, x in bad.items():
        assert _host_prefill({**t, n: x}) is None, n
        with pytest.raises((TypeError, ValueError)):
            gdn.prefill_run(**{**t, n: x})
    out = torch.empty_like(t["v"])
    overlapping = torch.empty(t["state"].numel() + 128, device=hip_device)
    overlapping[:t["state"].numel()].copy_(t["state"].view(-1))
    s0 = overlapping[:t["state"].numel()].view(t["state"].shape)
    s1 = overlapping[128:].view(t["state"].shape)
    assert _host_prefill({**t, "state": s0}, False, out, s1) is None
    with pytest.raises(ValueError):
        gdn.kernel_prefill_hip(**{**t, "state": s0}, output=out, new_state=s1)
    d = _dev(make_inputs(2, 4, 8, seed=822), hip_device)
    names = ("q", "k", "v", "state", "A_log", "a", "dt_bias", "b", "scale")
    for n, x in {"state": d["state"].half(), "q": d["q"][:, :, :, :64], "b": d["b"].float(),
                 "A_log": d["A_log"].cpu()}.items():
        args = [{**d, n: x}[m] for m in names]
        assert _lib.bound_host.decode_run(*args, False) is None, n
        with pytest.raises((TypeError, ValueError)):
            gdn.run(*args)


@pytest.mark.parametrize("lens", [[6], [64], [65, 7]])
def test_captured_prefill_replays(lens, hip_device):
    """A prefill captured by torch after one eager call (which binds the
    native path): replays over new inputs equal the eager results."""
    _announce(f"captured prefill lens={lens}")
    H, HV = 4, 8
    t = _dev(make_prefill_inputs(lens, H, HV, seed=831), hip_device)
    out, st = torch.empty_like(t["v"]), torch.empty_like(t["state"])
    gdn.kernel_prefill_hip(**t, output=out, new_state=st)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        gdn.kernel_prefill_hip(**t, output=out, new_state=st)
    for rnd in range(3):
        fresh = _dev(make_prefill_inputs(lens, H, HV, seed=840 + rnd), hip_device)
        for n in ("q", "k", "v", "state", "a", "b"):
            t[n].copy_(fresh[n])
        graph.replay()
        torch.cuda.synchronize()
        ref_o, ref_s = gdn.prefill_run(**t)
        torch.cuda.synchronize()
        assert torch.equal(out, ref_o) and torch.equal(st, ref_s), rnd


@pytest.mark.parametrize("lens", [[6], [64], [65, 7]])
@pytest.mark.parametrize("native", [False, True])
def test_lazily_cloned_destinations_get_their_own_memory(lens, native, hip_device):
    """An output and a new state that are lazy clones share memory with their
    originals until written: the call writes the clones alone."""
    _announce(f"lazy clones as destinations lens={lens} native={native}")
    H, HV = 4, 8
    t = _dev(make_prefill_inputs(lens, H, HV, seed=851), hip_device)
    ref_o, ref_s = gdn.prefill_run(**t)
    state, base = t["state"].clone(), torch.zeros_like(t["v"])
    out, st = torch._lazy_clone(base), torch._lazy_clone(t["state"])
    if native:
        assert _host_prefill(t, False, out, st) == 0
    else:
        pmod._prefill_checked(t["q"], t["k"], t["v"], t["state"], t["A_log"], t["a"],
                              t["dt_bias"], t["b"], t["cu_seqlens"], t["scale"], out, st, False)
    torch.cuda.synchronize()
    assert torch.equal(out, ref_o) and torch.equal(st, ref_s)
    assert torch.equal(t["state"], state) and not base.any()
