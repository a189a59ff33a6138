"""GPU parity tests of the varlen chunked prefill kernel (through the C ABI)
against the CPU oracle, plus size-independent properties at full size."""
import ctypes

import numpy as np
import pytest
import torch

from gdn_kernel_amd import _lib, binding, workloads
from gdn_kernel_amd.workloads import Heads, to_numpy
from oracle import gdn_oracle as O
from tests.conftest import assert_close
from tests.gpu_util import (OUT_ATOL, OUT_RTOL, STATE_ATOL, STATE_RTOL, host, oracle_prefill,
                            run_decode, run_prefill, say)

pytestmark = pytest.mark.gpu

CASES = {
    "one_chunk": [64],
    "one_token": [1],
    "short": [63],
    "partial": [65],
    "two_seqs": [130, 7],
    "ragged_empty": [0, 5, 64, 0, 200],
    "long": [300],
}


@pytest.mark.parametrize("case", list(CASES))
@pytest.mark.parametrize("gate", ["baseline", "slow"])
def test_prefill_matches_oracle(gpu, case, gate):
    lens = CASES[case]
    say(f"prefill parity case={case} lens={lens} gate={gate}")
    p = workloads.prefill_inputs(lens, seed=len(lens) * 7 + sum(lens), gate=gate,
                                 state_scale=0.5 if gate == "slow" else 0.05)
    o_ref, s_ref = oracle_prefill(p)
    out, ns = run_prefill(p, gpu)
    torch.cuda.synchronize()
    assert_close(host(out), o_ref, OUT_RTOL, OUT_ATOL, "output")
    assert_close(host(ns), s_ref, STATE_RTOL, STATE_ATOL, "new_state")


@pytest.mark.parametrize("cu_dtype", [torch.int32, torch.int64])
def test_prefill_null_state_and_cu_dtypes(gpu, cu_dtype):
    say(f"prefill null state cu={cu_dtype}")
    p = workloads.prefill_inputs([70, 3, 0], seed=11, gate="slow", with_state=False,
                                 cu_dtype=cu_dtype)
    o_ref, s_ref = oracle_prefill(p)
    out, ns = run_prefill(p, gpu)
    torch.cuda.synchronize()
    assert_close(host(out), o_ref, OUT_RTOL, OUT_ATOL, "output")
    assert_close(host(ns), s_ref, STATE_RTOL, STATE_ATOL, "new_state")
    assert not host(ns)[2].any()                      # empty sequence, zero initial state


@pytest.mark.parametrize("lens", [[100, 0, 20], [100, 20]])   # 96 chains split 2 ways; 64 split 4 ways
def test_prefill_in_place(gpu, lens):
    say(f"prefill in place lens={lens}")
    p = workloads.prefill_inputs(lens, seed=12, gate="slow", state_scale=0.5)
    o1, s1 = run_prefill(p, gpu, in_place=False)
    o2, s2 = run_prefill(p, gpu, in_place=True)
    torch.cuda.synchronize()
    assert torch.equal(o1, o2) and torch.equal(s1, s2)


@pytest.mark.parametrize("hq,hk,hv", [(8, 8, 32), (32, 32, 32), (2, 4, 8)])
def test_prefill_head_ratios(gpu, hq, hk, hv):
    say(f"prefill heads hq={hq} hk={hk} hv={hv}")
    p = workloads.prefill_inputs([90, 17], Heads(hq, hk, hv), seed=13, gate="slow",
                                 state_scale=0.5)
    o_ref, s_ref = oracle_prefill(p)
    out, ns = run_prefill(p, gpu)
    torch.cuda.synchronize()
    assert_close(host(out), o_ref, OUT_RTOL, OUT_ATOL, "output")
    assert_close(host(ns), s_ref, STATE_RTOL, STATE_ATOL, "new_state")


def test_prefill_sequential_definition(gpu):
    """Against the token-by-token definition directly (not only the chunk form)."""
    say("prefill vs sequential definition")
    p = workloads.prefill_inputs([150, 40], Heads(4, 4, 8), seed=14, gate="slow",
                                 state_scale=0.5)
    o_ref, s_ref = oracle_prefill(p, chunked=False)
    out, ns = run_prefill(p, gpu)
    torch.cuda.synchronize()
    assert_close(host(out), o_ref, OUT_RTOL, OUT_ATOL, "output")
    assert_close(host(ns), s_ref, STATE_RTOL, STATE_ATOL, "new_state")


def test_prefill_T1_equals_decode_kernel(gpu):
    say("prefill T=1 vs decode kernel")
    p = workloads.prefill_inputs([1] * 5, seed=15, gate="slow", state_scale=0.5)
    out, ns = run_prefill(p, gpu)
    w = {k: p[k][:, None] if k in ("q", "k", "v", "a", "b") else p[k]
         for k in ("q", "k", "v", "a", "b", "A_log", "dt_bias", "state", "scale")}
    o2, s2 = run_decode(w, gpu, in_place=False)
    torch.cuda.synchronize()
    assert_close(host(out), host(o2[:, 0]), OUT_RTOL, OUT_ATOL, "output")
    assert_close(host(ns), host(s2), STATE_RTOL, STATE_ATOL, "state")


def test_prefill_golden_fixture(gpu):
    say("prefill golden fixture")
    from tests.golden import path
    fx = np.load(path("prefill_small.npz"))
    bf = lambda n: torch.from_numpy(fx[n]).to(gpu).view(torch.bfloat16)
    state = torch.from_numpy(O.bits_to_f32(fx["state"])).to(gpu)
    out = torch.empty((fx["v"].shape[0], fx["v"].shape[1], 128), dtype=torch.bfloat16, device=gpu)
    ns = torch.empty_like(state)
    binding.prefill_kernel(bf("q"), bf("k"), bf("v"), state, torch.from_numpy(fx["A_log"]).to(gpu),
                           bf("a"), torch.from_numpy(fx["dt_bias"]).to(gpu), bf("b"),
                           torch.from_numpy(fx["cu_seqlens"]).to(gpu), float(fx["scale"]), out, ns)
    torch.cuda.synchronize()
    assert_close(host(out), fx["out_ref"], OUT_RTOL, OUT_ATOL, "output")
    assert_close(host(ns), fx["state_ref"], STATE_RTOL, STATE_ATOL, "new_state")


def _split_run(p, cut, gpu):
    """Run a single sequence in two calls, handing the state over at ``cut``."""
    d = {k: (v.to(gpu) if isinstance(v, torch.Tensor) else v) for k, v in p.items()}
    T = d["q"].shape[0]
    out = torch.empty((T, d["v"].shape[1], 128), dtype=torch.bfloat16, device=gpu)
    st = d["state"].clone() if d["state"] is not None else torch.zeros(
        (1, d["v"].shape[1], 128, 128), device=gpu)
    for s, e in ((0, cut), (cut, T)):
        cu = torch.tensor([0, e - s], dtype=torch.int32, device=gpu)
        binding.prefill_kernel(d["q"][s:e], d["k"][s:e], d["v"][s:e], st, d["A_log"], d["a"][s:e],
                               d["dt_bias"], d["b"][s:e], cu, d["scale"], out[s:e], st)
    return out, st


def test_prefill_config3_full_size(gpu):
    """BASELINE config 3 (T=4096, one sequence, zero initial state): the full output and
    the final state against the oracle, and the kernel split in two calls at a chunk
    boundary and off a chunk boundary (state hand-off) against the one-call result."""
    say("prefill config3 full size")
    p = workloads.config(3)
    out, ns = run_prefill(p, gpu)
    o_ref, s_ref = oracle_prefill(p)
    torch.cuda.synchronize()
    assert_close(host(out), o_ref, OUT_RTOL, OUT_ATOL, "output")
    assert_close(host(ns), s_ref, STATE_RTOL, STATE_ATOL, "new_state")
    for cut in (2048, 1000):
        o2, s2 = _split_run(p, cut, gpu)
        torch.cuda.synchronize()
        assert_close(host(o2), host(out), OUT_RTOL, OUT_ATOL, f"split@{cut} output")
        assert_close(host(s2), host(ns), STATE_RTOL, STATE_ATOL, f"split@{cut} state")


def test_prefill_config4_full_size(gpu):
    """BASELINE config 4 (32 sequences, 32768 tokens, int32 cu_seqlens, random initial
    states): every output token and every sequence's final state against the oracle on
    the whole packed batch; the longest and the shortest sequence run alone give the
    packed results bit for bit."""
    say("prefill config4 full size")
    p = workloads.config(4)
    lens = p["lengths"]
    assert min(lens) < 64 and sum(lens) == 32768
    out, ns = run_prefill(p, gpu)
    o_ref, s_ref = oracle_prefill(p)
    torch.cuda.synchronize()
    assert_close(host(out), o_ref, OUT_RTOL, OUT_ATOL, "output")
    assert_close(host(ns), s_ref, STATE_RTOL, STATE_ATOL, "new_state")
    cu = p["cu_seqlens"].tolist()
    order = np.argsort(lens)
    for i in (int(order[-1]), int(order[0])):
        s, e = cu[i], cu[i + 1]
        sub = {k: (p[k][s:e] if k in ("q", "k", "v", "a", "b") else p[k])
               for k in ("q", "k", "v", "a", "b", "A_log", "dt_bias", "scale")}
        sub["state"] = p["state"][i:i + 1]
        sub["cu_seqlens"] = torch.tensor([0, e - s], dtype=torch.int32)
        o1, s1 = run_prefill(sub, gpu)
        torch.cuda.synchronize()
        assert torch.equal(o1, out[s:e]) and torch.equal(s1[0], ns[i]), f"seq {i} packed != alone"


@pytest.mark.parametrize("lens", [[1, 63, 64, 65, 130], [300]])
@pytest.mark.parametrize("state_scale", [0.05, 0.5])
def test_prefill_edge_gates(gpu, lens, state_scale):
    """The gate prologue's edge branches against the oracle: softplus arguments above 20
    (its linear branch), saturated beta (b = +-12, +-30) and A_log from -12 (no decay) to
    4 (e^4 per unit of softplus: the state is wiped by any token with a > 20), per v-head.
    Fast-decay chunks take the log-gate sums to ~1e5 in magnitude while the decays that
    matter come from differences below 1e2: the kernel sums them in fp64.  Both batches run
    as one kernel; the single 300-token sequence (32 chains) also on the two-kernel path,
    with a workspace."""
    say(f"prefill edge gates lens={lens} state_scale={state_scale}")
    p = workloads.prefill_inputs(lens, seed=41, gate="edge", state_scale=state_scale)
    x = to_numpy(p["a"]) + to_numpy(p["dt_bias"])
    assert (x > 20).any() and (np.abs(to_numpy(p["b"])) >= 12).any()
    assert _dropin_windows(p)[0] == 0
    o_ref, s_ref = oracle_prefill(p)
    out, ns = run_prefill(p, gpu)
    torch.cuda.synchronize()
    if len(lens) == 1:
        o2, s2 = _prefill_capi(p, gpu, workspace=True)
        assert torch.equal(o2, out) and torch.equal(s2, ns), "workspace path differs from one kernel"
    assert_close(host(out), o_ref, OUT_RTOL, OUT_ATOL, "output")
    assert_close(host(ns), s_ref, STATE_RTOL, STATE_ATOL, "new_state")


@pytest.mark.parametrize("lens,heads", [([1500], Heads(4, 4, 8)), ([2002], Heads(16, 16, 32))])
def test_prefill_no_decay_precision_envelope(gpu, lens, heads):
    """Long chains with no decay at all (A_log = -12, g = 1 to fp32 precision) and
    saturated beta: the state-path operands are bf16 hi + lo pairs (about 16 significant
    bits), so the state error does not decay away and settles at about 5e-6 of the
    head's largest state element.  Near-zero elements of a state whose entries reach ~3
    can then exceed the strict bound (atol 1e-5 + rtol 1e-3 |ref|) by tens of percent.  This
    test pins that envelope: the outputs within the strict tolerance, and every state
    element within 2e-5 x the largest |state| of its head (besides rtol 1e-3).  With no
    decay a wrong gate or tile anywhere in the chain stays in the final state: the second
    case (one sequence of 2,002 tokens, 32 chains) runs gdn_prefill's two kernels, where a
    chunk image copied out of LDS while the next chunk's gates were being written to the
    same slots gives a state error of about 4e4 x the bound."""
    say(f"prefill no-decay precision envelope lens={lens} heads={heads}")
    p = workloads.prefill_inputs(lens, heads, seed=43, gate="edge", state_scale=0.5)
    p["A_log"] = torch.full((heads.hv,), -12.0)
    assert _dropin_windows(p) == (1, 0)
    o_ref, s_ref = oracle_prefill(p)
    out, ns = run_prefill(p, gpu)
    torch.cuda.synchronize()
    assert_close(host(out), o_ref, OUT_RTOL, OUT_ATOL, "output")
    got = host(ns)
    scale = np.abs(s_ref).max(axis=(2, 3), keepdims=True)
    err = np.abs(got - s_ref)
    bound = 2e-5 * scale + STATE_RTOL * np.abs(s_ref)
    assert (err <= bound).all(), f"max err / bound = {(err / bound).max():.3f}"
    assert (err / scale).max() < 2e-5


def test_prefill_split_variants_bitwise(gpu):
    """Chains are split over 8, 4, 2 or 1 workgroups depending on how many (sequence,
    v-head) chains the batch has.  Every split does the same per-row arithmetic, so
    padding a batch with empty sequences (more chains, a smaller split) must not change
    a single bit of the real sequences' outputs and states; the smallest batch is also
    checked against the oracle."""
    heads = Heads(4, 4, 8)
    real = [150, 64, 7]
    p = workloads.prefill_inputs(real + [0] * 17, heads, seed=16, gate="slow", state_scale=0.5)
    results = []
    for n in (3, 5, 13, 20):          # 24, 40, 104, 160 chains: splits 8, 4, 2, 1 on 256 CUs
        say(f"prefill split variants: {n} sequences ({n * heads.hv} chains)")
        sub = dict(p)
        sub["cu_seqlens"] = p["cu_seqlens"][:n + 1]
        sub["state"] = p["state"][:n]
        out, ns = run_prefill(sub, gpu)
        torch.cuda.synchronize()
        results.append((out, ns[:len(real)]))
        if n == 3:
            o_ref, s_ref = oracle_prefill(sub)
            assert_close(host(out), o_ref, OUT_RTOL, OUT_ATOL, "output")
            assert_close(host(ns), s_ref, STATE_RTOL, STATE_ATOL, "new_state")
        else:
            assert not host(ns[len(real):] - sub["state"][len(real):].to(gpu)).any(), \
                "empty sequences must pass their state through"
    for i, (o, s) in enumerate(results[1:], 1):
        assert torch.equal(o, results[0][0]), f"output differs between splits (run {i})"
        assert torch.equal(s, results[0][1]), f"state differs between splits (run {i})"


def test_prefill_more_sequences_than_the_sorted_schedule(gpu):
    """More than 1,024 sequences: workgroups take sequences in natural order instead
    of longest first.  Mostly empty sequences keep the oracle cheap."""
    rng = np.random.default_rng(17)
    lens = [0] * 1030
    for i in rng.choice(1030, 24, replace=False):
        lens[i] = int(rng.integers(1, 140))
    say(f"prefill {len(lens)} sequences, {sum(lens)} tokens")
    p = workloads.prefill_inputs(lens, Heads(2, 2, 4), seed=17, gate="slow", state_scale=0.5)
    o_ref, s_ref = oracle_prefill(p)
    out, ns = run_prefill(p, gpu)
    torch.cuda.synchronize()
    assert_close(host(out), o_ref, OUT_RTOL, OUT_ATOL, "output")
    assert_close(host(ns), s_ref, STATE_RTOL, STATE_ATOL, "new_state")


@pytest.mark.parametrize("cu_dtype", [torch.int32, torch.int64])
def test_prefill_malformed_cu_seqlens_are_clamped(gpu, cu_dtype):
    """Offsets are clamped on the device: sequence i covers [clamp(cu[i], 0, T),
    clamp(cu[i+1], start, T)).  cu = [0, 40, 20, 500] with T = 100 gives [0, 40),
    an empty sequence and [20, 100).  Tokens 20..39 belong to two sequences, so only
    the other outputs and the three final states are compared."""
    say(f"prefill malformed cu_seqlens {cu_dtype}")
    T = 100
    p = workloads.prefill_inputs([T], Heads(2, 2, 4), seed=18, gate="slow", state_scale=0.5)
    state = 0.5 * torch.randn((3, 4, 128, 128), generator=torch.Generator().manual_seed(18))
    bad = dict(p, state=state, cu_seqlens=torch.tensor([0, 40, 20, 500], dtype=cu_dtype))
    out, ns = run_prefill(bad, gpu)
    torch.cuda.synchronize()
    for i, (s, e) in ((0, (0, 40)), (2, (20, 100))):
        sub = {k: (p[k][s:e] if k in ("q", "k", "v", "a", "b") else p[k])
               for k in ("q", "k", "v", "a", "b", "A_log", "dt_bias", "scale")}
        sub["state"] = state[i:i + 1]
        sub["cu_seqlens"] = torch.tensor([0, e - s], dtype=torch.int32)
        o_ref, s_ref = oracle_prefill(sub)
        keep = slice(0, 20) if i == 0 else slice(20, 80)   # tokens owned by one sequence only
        assert_close(host(out[s:e])[keep], o_ref[keep], OUT_RTOL, OUT_ATOL, f"seq {i} output")
        assert_close(host(ns[i]), s_ref[0], STATE_RTOL, STATE_ATOL, f"seq {i} state")
    assert torch.equal(ns[1].cpu(), state[1]), "the empty sequence passes its state through"


@pytest.mark.parametrize("with_state", [True, False])
def test_prefill_no_tokens(gpu, with_state):
    """T = 0: every sequence is empty; new_state is the initial state (or zeros)."""
    say(f"prefill T=0 with_state={with_state}")
    p = workloads.prefill_inputs([0, 0, 0], Heads(2, 2, 4), seed=19, with_state=with_state)
    out, ns = run_prefill(p, gpu)
    torch.cuda.synchronize()
    assert out.numel() == 0
    ref = p["state"] if with_state else torch.zeros_like(ns.cpu())
    assert torch.equal(ns.cpu(), ref)


def _prefill_fault_injection(p, gpu, spin_limit, ready_chunks, workspace=False):
    """gdn_prefill_fault_injection (one kernel), or with `workspace`
    gdn_prefill_fault_injection_with_workspace, through the C ABI; returns (output,
    new_state, aborts)."""
    d = {k: (v.to(gpu) if isinstance(v, torch.Tensor) else v) for k, v in p.items()}
    T, Hq = d["q"].shape[0], d["q"].shape[1]
    Hk, Hv = d["k"].shape[1], d["v"].shape[1]
    cu = d["cu_seqlens"]
    N = cu.numel() - 1
    out = torch.full((T, Hv, 128), float("nan"), device=gpu, dtype=torch.bfloat16)
    ns = torch.full((N, Hv, 128, 128), float("nan"), device=gpu, dtype=torch.float32)
    aborts = torch.zeros(1, device=gpu, dtype=torch.int32)
    cu_code = _lib.GDN_INDEX_INT32 if cu.dtype == torch.int32 else _lib.GDN_INDEX_INT64
    ptr = lambda t: None if t is None else t.data_ptr()
    args = [ptr(d["q"]), ptr(d["k"]), ptr(d["v"]), ptr(d["state"]), ptr(d["A_log"]), ptr(d["a"]),
            ptr(d["dt_bias"]), ptr(d["b"]), cu.data_ptr(), cu_code, N, T, d["scale"], ptr(out), ptr(ns),
            Hq, Hk, Hv, 128, 128]
    hooks = [spin_limit, ready_chunks, ptr(aborts), torch.cuda.current_stream(gpu).cuda_stream]
    lib = _lib.load()
    if workspace:
        nbytes = lib.gdn_prefill_workspace_size(N, T, Hv)
        assert nbytes > 0, "expected a batch that the two-kernel path serves"
        ws = torch.full((nbytes,), 0xFF, device=gpu, dtype=torch.uint8)
        _lib.check(lib.gdn_prefill_fault_injection_with_workspace(*args, ptr(ws), nbytes, *hooks))
        torch.cuda.synchronize()
    else:
        _lib.check(lib.gdn_prefill_fault_injection(*args, *hooks))
    return out, ns, aborts


def _dropin_windows(p):
    """How gdn_prefill runs the batch: (windows of the two-kernel path, 0 for one kernel;
    whether it yields to another stream)."""
    yields = ctypes.c_int32(-1)
    n = _lib.load().gdn_prefill_dropin_windows(p["cu_seqlens"].numel() - 1, p["q"].shape[0], p["v"].shape[1],
                                               ctypes.byref(yields))
    return n, yields.value


def _prefill_capi(p, gpu, workspace, ws=None, nbytes=None):
    """gdn_prefill, or gdn_prefill_with_workspace with a workspace of exactly the
    reported size (or the given buffer), through the C ABI; returns (output, new_state)."""
    d = {k: (v.to(gpu) if isinstance(v, torch.Tensor) else v) for k, v in p.items()}
    T, Hq = d["q"].shape[0], d["q"].shape[1]
    Hk, Hv = d["k"].shape[1], d["v"].shape[1]
    cu = d["cu_seqlens"]
    N = cu.numel() - 1
    out = torch.full((T, Hv, 128), float("nan"), device=gpu, dtype=torch.bfloat16)
    ns = torch.full((N, Hv, 128, 128), float("nan"), device=gpu, dtype=torch.float32)
    cu_code = _lib.GDN_INDEX_INT32 if cu.dtype == torch.int32 else _lib.GDN_INDEX_INT64
    ptr = lambda t: None if t is None else t.data_ptr()
    args = [ptr(d["q"]), ptr(d["k"]), ptr(d["v"]), ptr(d["state"]), ptr(d["A_log"]), ptr(d["a"]),
            ptr(d["dt_bias"]), ptr(d["b"]), cu.data_ptr(), cu_code, N, T, d["scale"], ptr(out),
            ptr(ns), Hq, Hk, Hv, 128, 128]
    lib = _lib.load()
    stream = torch.cuda.current_stream(gpu).cuda_stream
    if workspace:
        if ws is None:
            nbytes = lib.gdn_prefill_workspace_size(N, T, Hv)
            assert nbytes > 0, "expected a batch that the two-kernel path serves"
            ws = torch.full((nbytes,), 0xFF, device=gpu, dtype=torch.uint8)
        rc = lib.gdn_prefill_with_workspace(*args, ws.data_ptr(), nbytes, stream)
    else:
        rc = lib.gdn_prefill(*args, stream)
    _lib.check(rc)
    torch.cuda.synchronize()
    return out, ns


@pytest.mark.parametrize("lens,heads", [
    ([300], Heads(16, 16, 32)),                  # 32 chains, each split over 8 workgroups
    ([150, 64, 7, 0], Heads(4, 4, 8)),           # ragged, an empty sequence
    ([150, 64, 7, 0, 65, 200], Heads(4, 4, 8)),  # 48 chains: split 4 ways (two 16-row consumers)
    ([130, 2100], Heads(16, 16, 32)),            # 64 chains, split 4 ways
    ([1, 2, 63, 64, 129], Heads(2, 2, 4)),       # boundary lengths
    ([700, 1300], Heads(8, 8, 16)),              # 32 chains of many chunks
    ([1000], Heads(16, 8, 32)),                  # distinct q and k head ratios, split 8 ways
    ([3000, 2000], Heads(16, 16, 32)),           # 64 chains over 97 MB of images
])
def test_prefill_two_kernel_path(gpu, lens, heads):
    """Batches of at most 64 chains with a workspace: a first kernel prepares every
    chunk's T~, P and gates (all chunks at once) and the state pass copies them instead
    of recomputing them in each of a chain's 4 or 8 slices; split 8 ways, four consumer
    waves share each slice's chunk tokens.  Every value comes from the same operations in
    the same order, so the results equal one kernel's bit for bit (launched by the testing
    entry point, which has no two-kernel path of its own), as do gdn_prefill's, whichever it
    runs; both match the oracle.  The workspace starts as 0xFF bytes, so a chunk image that
    the first kernel did not write would show."""
    say(f"prefill two-kernel path lens={lens} heads={heads}")
    p = workloads.prefill_inputs(lens, heads, seed=22, gate="slow", state_scale=0.5)
    o0, s0, _ = _prefill_fault_injection(p, gpu, 0, 0)
    o1, s1 = _prefill_capi(p, gpu, workspace=False)
    o2, s2 = _prefill_capi(p, gpu, workspace=True)
    assert torch.equal(o0, o2) and torch.equal(s0, s2), "workspace path differs from one kernel"
    assert torch.equal(o1, o2) and torch.equal(s1, s2), "workspace path differs from gdn_prefill"
    o_ref, s_ref = oracle_prefill(p)
    assert_close(host(o2), o_ref, OUT_RTOL, OUT_ATOL, "output")
    assert_close(host(s2), s_ref, STATE_RTOL, STATE_ATOL, "new_state")


@pytest.mark.parametrize("seed", [0, 4, 5, 9, 24, 28, 30])   # heads 4, 8, 16 and 32 v-heads, 1-3 sequences
def test_prefill_dropin_random_long_batches(gpu, seed):
    """Seeded random batches that gdn_prefill runs on its two-kernel path (at most 64
    chains whose sequences average at least 1,024 tokens, images within its scratch):
    1-3 sequences of 1-2,000 tokens topped up to that average, random head layouts, gate
    regime, initial states and cu_seqlens dtype.  gdn_prefill equals
    gdn_prefill_with_workspace and one kernel bit for bit, all match the oracle, and no
    hand-off gives up."""
    rng = np.random.default_rng(3000 + seed)
    hq, hk, hv = [(16, 16, 32), (8, 8, 16), (4, 8, 8), (2, 2, 4), (4, 4, 16)][int(rng.integers(0, 5))]
    n = min(int(rng.integers(1, 4)), 64 // hv)
    lens = [int(rng.integers(1, 2001)) for _ in range(n)]
    short = 1024 * n - sum(lens)
    if short > 0:
        lens[int(rng.integers(0, n))] += short
    gate = "slow" if rng.random() < 0.5 else "baseline"
    with_state = bool(rng.random() < 0.7)
    cu_dtype = torch.int64 if rng.random() < 0.5 else torch.int32
    say(f"prefill drop-in random long batch seed={seed} lens={lens} heads=({hq},{hk},{hv}) gate={gate} "
        f"state={with_state} cu={cu_dtype}")
    p = workloads.prefill_inputs(lens, Heads(hq, hk, hv), seed=4000 + seed, gate=gate,
                                 state_scale=0.5 if gate == "slow" else 0.05, with_state=with_state,
                                 cu_dtype=cu_dtype)
    binding.prefill_giveups(reset=True)
    assert _dropin_windows(p) == (1, 0)
    o0, s0, _ = _prefill_fault_injection(p, gpu, 0, 0)
    o1, s1 = _prefill_capi(p, gpu, workspace=False)
    o2, s2 = _prefill_capi(p, gpu, workspace=True)
    assert torch.equal(o1, o2) and torch.equal(s1, s2), "gdn_prefill differs from gdn_prefill_with_workspace"
    assert torch.equal(o0, o1) and torch.equal(s0, s1), "gdn_prefill differs from one kernel"
    o_ref, s_ref = oracle_prefill(p)
    assert_close(host(o1), o_ref, OUT_RTOL, OUT_ATOL, "output")
    assert_close(host(s1), s_ref, STATE_RTOL, STATE_ATOL, "new_state")
    assert binding.prefill_giveups() == 0


@pytest.mark.parametrize("lens,heads", [
    ([int(x) for x in np.random.default_rng(91).integers(0, 131, 64)], Heads(1, 1, 1)),  # 64 sequences, one head
    ([65, 0, 1, 64, 127], Heads(3, 1, 3)),          # odd heads: a prep workgroup spans two chunks
    ([129, 700], Heads(2, 8, 16)),                  # distinct q and k ratios
])
def test_prefill_prep_kernel_edges(gpu, lens, heads):
    """The prep kernel (a wave per chunk-head) where its indexing can go wrong: many
    sequences, odd head counts, ragged and empty sequences.  Bit for bit one kernel, and
    within tolerance of the oracle."""
    say(f"prefill prep kernel edges lens={lens} heads={heads}")
    p = workloads.prefill_inputs(lens, heads, seed=92, gate="slow", state_scale=0.5)
    o1, s1, _ = _prefill_fault_injection(p, gpu, 0, 0)
    o2, s2 = _prefill_capi(p, gpu, workspace=True)
    assert torch.equal(o1, o2) and torch.equal(s1, s2)
    o_ref, s_ref = oracle_prefill(p)
    assert_close(host(o2), o_ref, OUT_RTOL, OUT_ATOL, "output")
    assert_close(host(s2), s_ref, STATE_RTOL, STATE_ATOL, "new_state")


def test_prefill_two_kernels_overlapping_offsets(gpu):
    """Malformed offsets on the two-kernel path: cu = [0, 200, 0, 200, 90] with T = 200
    gives [0, 200), an empty sequence, [0, 200) again and an empty one: eight chunks, more
    than any valid offsets of four sequences give (seven).  Both final states are those of
    the 200 tokens; the outputs belong to two sequences and are not compared."""
    say("prefill two kernels, overlapping offsets")
    heads = Heads(2, 2, 4)
    p = workloads.prefill_inputs([200], heads, seed=93, gate="slow", state_scale=0.5)
    state = 0.5 * torch.randn((4, 4, 128, 128), generator=torch.Generator().manual_seed(93))
    bad = dict(p, state=state, cu_seqlens=torch.tensor([0, 200, 0, 200, 90], dtype=torch.int32))
    _, ns = _prefill_capi(bad, gpu, workspace=True)
    for i in (0, 2):
        _, s_ref = oracle_prefill(dict(p, state=state[i:i + 1], cu_seqlens=torch.tensor([0, 200], dtype=torch.int32)))
        assert_close(host(ns[i]), s_ref[0], STATE_RTOL, STATE_ATOL, f"seq {i} state")
    assert torch.equal(ns[1].cpu(), state[1]) and torch.equal(ns[3].cpu(), state[3])


def test_prefill_workspace_reuse(gpu):
    """One workspace buffer, not cleared between calls, serves two different few-chain
    batches in turn (the larger first, then a smaller one whose images overlay the
    first's, then the larger again): every call equals gdn_prefill bit for bit, so no
    result depends on images left by an earlier call."""
    lib = _lib.load()
    big = workloads.prefill_inputs([700, 300], Heads(8, 8, 16), seed=23, gate="slow", state_scale=0.5)
    small = workloads.prefill_inputs([90, 0, 130], Heads(4, 4, 8), seed=24, gate="slow", state_scale=0.5)
    need = [lib.gdn_prefill_workspace_size(len(p["lengths"]), p["q"].shape[0], p["v"].shape[1]) for p in (big, small)]
    assert min(need) > 0
    ws = torch.full((max(need),), 0x5A, device=gpu, dtype=torch.uint8)
    for name, p, nb in (("big", big, need[0]), ("small", small, need[1]), ("big", big, need[0])):
        say(f"prefill workspace reuse: {name} batch")
        ref_o, ref_s = _prefill_capi(p, gpu, workspace=False)
        o, s = _prefill_capi(p, gpu, workspace=True, ws=ws, nbytes=nb)
        assert torch.equal(o, ref_o) and torch.equal(s, ref_s), f"{name}: workspace path differs"


@pytest.mark.giveups_expected
@pytest.mark.parametrize("heads,split", [(Heads(16, 16, 32), 2), (Heads(8, 8, 16), 4), (Heads(4, 4, 8), 8)])
def test_prefill_bounded_waits(gpu, heads, split):
    """The hand-off failure path, forced from the host.  With the testing hooks off
    the entry point is gdn_prefill bit for bit and nothing gives up.  With the
    producers signalling only their first chunk and a 2,000-poll wait limit, every
    workgroup of a sequence with two or more chunks has a consumer wait that can only
    give up: the launch still completes (every wait is bounded), the give-ups are
    counted both by the hook counter and by the device counter that
    gdn_prefill_giveups reports, every output and final-state element of the affected
    sequences is NaN, the one-chunk sequence's results are untouched, and the next
    normal launch is exact again.  With 32 v-heads the 96 chains split 2 ways (four
    producer waves per workgroup); with 16 the 48 chains split 4 ways (six, pipelined);
    with 8 the 24 chains split 8 ways (seven, pipelined)."""
    lens = [300, 130, 40]             # 5, 3 and 1 chunks
    p = workloads.prefill_inputs(lens, heads, seed=21, gate="slow", state_scale=0.5)
    binding.prefill_giveups(reset=True)
    say("prefill bounded waits: hooks off")
    o0, s0, a0 = _prefill_fault_injection(p, gpu, 0, 0)
    o1, s1 = run_prefill(p, gpu)
    torch.cuda.synchronize()
    assert int(a0.item()) == 0 and binding.prefill_giveups() == 0
    assert torch.equal(o0, o1) and torch.equal(s0, s1)
    say("prefill bounded waits: chunk-ready signals stop after chunk 0, 2000-poll limit")
    o2, s2, a2 = _prefill_fault_injection(p, gpu, 2000, 1)
    torch.cuda.synchronize()
    waiting_wgs = 2 * heads.hv * split  # sequences with >= 2 chunks x v-heads x workgroups per chain
    n = int(a2.item())
    assert waiting_wgs <= n <= waiting_wgs * 8, n
    assert binding.prefill_giveups(reset=True) == n, "the device counter must see every give-up"
    s, e = sum(lens[:2]), sum(lens)
    assert torch.isnan(o2[:s].float()).all() and torch.isnan(s2[:2]).all(), \
        "outputs and states of the sequences whose waits gave up must be NaN"
    assert torch.equal(o2[s:e], o1[s:e]) and torch.equal(s2[2], s1[2])
    say("prefill bounded waits: a normal launch afterwards")
    o3, s3 = run_prefill(p, gpu)
    torch.cuda.synchronize()
    assert torch.equal(o3, o1) and torch.equal(s3, s1)
    assert binding.prefill_giveups() == 0


@pytest.mark.giveups_expected
@pytest.mark.parametrize("heads,split", [(Heads(8, 8, 16), 4), (Heads(4, 4, 8), 8)])
def test_prefill_two_kernels_bounded_waits(gpu, heads, split):
    """The hand-off failure path of the state pass (48 chains split 4 ways: the general
    kernel's loader variant; 24 split 8 ways: the state kernel), forced from the host as in
    test_prefill_bounded_waits: with the waves that stage the chunks signalling only the
    first, every workgroup of a sequence of two or more chunks gives up, is counted, and
    leaves NaN in every output and final-state element it owns; the one-chunk sequence is
    untouched, and with the hooks off, before and after, nothing gives up."""
    lens = [300, 130, 40]             # 5, 3 and 1 chunks
    p = workloads.prefill_inputs(lens, heads, seed=23, gate="slow", state_scale=0.5)
    binding.prefill_giveups(reset=True)
    say(f"prefill two kernels bounded waits, split {split}: hooks off")
    o1, s1 = _prefill_capi(p, gpu, workspace=True)
    o0, s0, a0 = _prefill_fault_injection(p, gpu, 0, 0, workspace=True)
    assert int(a0.item()) == 0 and binding.prefill_giveups() == 0
    assert torch.equal(o0, o1) and torch.equal(s0, s1)
    say("prefill two kernels bounded waits: chunk-ready signals stop after chunk 0, 2000-poll limit")
    o2, s2, a2 = _prefill_fault_injection(p, gpu, 2000, 1, workspace=True)
    waiting_wgs = 2 * heads.hv * split  # sequences with >= 2 chunks x v-heads x workgroups per chain
    n = int(a2.item())
    assert waiting_wgs <= n <= waiting_wgs * 8, n
    assert binding.prefill_giveups(reset=True) == n, "the device counter must see every give-up"
    s, e = sum(lens[:2]), sum(lens)
    assert torch.isnan(o2[:s].float()).all() and torch.isnan(s2[:2]).all(), \
        "outputs and states of the sequences whose waits gave up must be NaN"
    assert torch.equal(o2[s:e], o1[s:e]) and torch.equal(s2[2], s1[2])
    say("prefill two kernels bounded waits: a normal launch afterwards")
    o3, s3 = _prefill_capi(p, gpu, workspace=True)
    assert torch.equal(o3, o1) and torch.equal(s3, s1)
    assert binding.prefill_giveups() == 0


@pytest.mark.parametrize("seed", range(6))
def test_prefill_random_batches(gpu, seed):
    """Seeded random batches against the oracle: 1-9 sequences with lengths drawn from
    the chunk-boundary values (0, 1, 63, 64, 65, 128) and uniformly up to 300, random
    head ratios, gate distribution and cu_seqlens dtype, with and without initial
    states.  The batch sizes land on different launch variants (chains split 1-8 ways)."""
    rng = np.random.default_rng(1000 + seed)
    n = int(rng.integers(1, 10))
    special = [0, 1, 63, 64, 65, 128]
    lens = [int(rng.choice(special)) if rng.random() < 0.4 else int(rng.integers(1, 301)) for _ in range(n)]
    hq, hk, hv = [(16, 16, 32), (8, 8, 32), (4, 8, 8), (2, 2, 8), (4, 4, 16)][int(rng.integers(0, 5))]
    gate = "slow" if rng.random() < 0.5 else "baseline"
    with_state = bool(rng.random() < 0.8)
    cu_dtype = torch.int64 if rng.random() < 0.5 else torch.int32
    say(f"prefill random batch seed={seed} lens={lens} heads=({hq},{hk},{hv}) gate={gate} "
        f"state={with_state} cu={cu_dtype}")
    p = workloads.prefill_inputs(lens, Heads(hq, hk, hv), seed=2000 + seed, gate=gate,
                                 state_scale=0.5 if gate == "slow" else 0.05, with_state=with_state,
                                 cu_dtype=cu_dtype)
    o_ref, s_ref = oracle_prefill(p)
    out, ns = run_prefill(p, gpu)
    torch.cuda.synchronize()
    assert_close(host(out), o_ref, OUT_RTOL, OUT_ATOL, "output")
    assert_close(host(ns), s_ref, STATE_RTOL, STATE_ATOL, "new_state")


def _heads_of(p, idx):
    """The inputs of v-heads ``idx`` alone, on the CPU (q/k heads likewise: the test's
    head counts are equal)."""
    gi = idx.to(p["q"].device)
    sub = {k: p[k][:, gi].cpu() for k in ("q", "k", "v", "a", "b")}
    sub.update({k: p[k][gi].cpu() for k in ("A_log", "dt_bias")})
    sub["state"] = None if p["state"] is None else p["state"][:, gi].cpu()
    sub["cu_seqlens"], sub["scale"] = p["cu_seqlens"].cpu(), p["scale"]
    return sub


def test_prefill_max_heads(gpu):
    """The largest head count the C ABI accepts (GDN_MAX_HEADS = 65,536 q, k and v heads),
    one 80-token sequence (a full chunk and a partial one): per-chunk row offsets are
    at their largest.  Every output element is written, and five heads at both ends and
    in the middle match the oracle run on those heads alone."""
    h = _lib.GDN_MAX_HEADS
    say(f"prefill max heads Hq=Hk=Hv={h} lens=[80]")
    p = workloads.prefill_inputs([80], Heads(h, h, h), seed=77, device=gpu, gate="slow",
                                 state_scale=0.5)
    out, ns = run_prefill(p, gpu)
    torch.cuda.synchronize()
    assert not torch.isnan(out).any() and not torch.isnan(ns).any()
    idx = torch.tensor([0, 1, h // 2 + 3, h - 2, h - 1])
    o_ref, s_ref = oracle_prefill(_heads_of(p, idx))
    assert_close(host(out[:, idx.to(gpu)]), o_ref, OUT_RTOL, OUT_ATOL, "output")
    assert_close(host(ns[:, idx.to(gpu)]), s_ref, STATE_RTOL, STATE_ATOL, "new_state")


def _persistent_lengths():
    rng = np.random.default_rng(77)
    return [0, 1, 63, 64, 65, 128, 129] + [int(x) for x in rng.integers(1, 300, 33)]


PERSISTENT_BATCHES = {
    # 40 sequences (zero, one and chunk-boundary lengths among them) of 8 v-heads:
    # 320 chains over 32 bins of 8 workgroups; no initial states
    "hv8_ragged": (_persistent_lengths(), Heads(4, 4, 8), False, False, torch.int32),
    # 64 sequences of 100 tokens, 32 v-heads: 2,048 chains over 8 bins, state
    # updated in place, int64 cu_seqlens
    "hv32_many_in_place": ([100] * 64, Heads(16, 16, 32), True, True, torch.int64),
    # 12 sequences, the 5 shortest empty: the bin whose first chain is empty, and an
    # empty chain after a non-empty one in another bin's list
    "empty_chains": ([300, 250, 200, 150, 100, 70, 65, 0, 0, 0, 0, 0], Heads(16, 16, 32), True, False,
                     torch.int32),
    # more than 64 sequences: lists in boustrophedon order over the longest-first
    # ranks; 200 sequences of 0-200 tokens, 32 v-heads (8 bins, 25 chains each)
    "hv32_200_seqs": ([int(x) for x in np.random.default_rng(78).integers(0, 201, 200)], Heads(16, 16, 32),
                      True, False, torch.int32),
    # 130 sequences of 0-300 tokens, 16 v-heads (16 bins, 8-9 chains each), in place
    "hv16_130_seqs": ([int(x) for x in np.random.default_rng(79).integers(0, 301, 130)], Heads(8, 8, 16),
                      True, True, torch.int64),
    # 80 sequences of 0-150 tokens, 4 v-heads (64 bins of 4 workgroups, 1-2 chains each)
    "hv4_80_seqs": ([int(x) for x in np.random.default_rng(80).integers(0, 151, 80)], Heads(2, 2, 4),
                    True, False, torch.int32),
    # distinct q and k head ratios (v-head h reads q-head h / 4 and k-head h / 2):
    # 20 sequences of 0-300 tokens, 32 v-heads
    "hq8_hk16_hv32": ([int(x) for x in np.random.default_rng(81).integers(0, 301, 20)], Heads(8, 16, 32),
                      True, False, torch.int32),
}


@pytest.mark.parametrize("case", list(PERSISTENT_BATCHES))
def test_prefill_persistent_batches(gpu, case):
    """Batches of more (sequence, v-head) chains than CUs (at most 1,024 sequences, Hv
    dividing the CU count) run one workgroup per CU, each through a list of chains:
    a longest-processing-time schedule up to 64 sequences, boustrophedon order over
    the longest-first ranks beyond.  Every output and final state against the
    oracle; three sequences run alone (a split launch) give the packed results bit
    for bit."""
    lens, heads, with_state, in_place, cu_dtype = PERSISTENT_BATCHES[case]
    say(f"prefill persistent batch {case}: {len(lens)} sequences, heads {heads}")
    p = workloads.prefill_inputs(lens, heads, seed=len(lens), gate="slow", state_scale=0.5,
                                 with_state=with_state, cu_dtype=cu_dtype)
    assert len(lens) * heads.hv > 256
    o_ref, s_ref = oracle_prefill(p)
    out, ns = run_prefill(p, gpu, in_place=in_place)
    torch.cuda.synchronize()
    assert_close(host(out), o_ref, OUT_RTOL, OUT_ATOL, "output")
    assert_close(host(ns), s_ref, STATE_RTOL, STATE_ATOL, "new_state")
    cu = p["cu_seqlens"].tolist()
    for i in (int(np.argmax(lens)), len(lens) // 2, len(lens) - 1):
        s, e = cu[i], cu[i + 1]
        sub = {k: (p[k][s:e] if k in ("q", "k", "v", "a", "b") else p[k])
               for k in ("q", "k", "v", "a", "b", "A_log", "dt_bias", "scale")}
        sub["state"] = None if p["state"] is None else p["state"][i:i + 1]
        sub["cu_seqlens"] = torch.tensor([0, e - s], dtype=torch.int32)
        o1, s1 = run_prefill(sub, gpu)
        torch.cuda.synchronize()
        assert torch.equal(o1, out[s:e]) and torch.equal(s1[0], ns[i]), f"seq {i} packed != alone"


@pytest.mark.giveups_expected
def test_prefill_persistent_bounded_waits(gpu):
    """The hand-off failure path of the persistent kernel, forced from the host: 12
    sequences of 2-5 chunks, 32 v-heads (384 chains, one workgroup per CU).  With the
    producers signalling only the first chunk of each chain and a 2,000-poll limit,
    each workgroup's first chain has a consumer wait that can only give up: the launch
    completes, the give-ups are counted by the hook counter and the device counter,
    every output and final state is NaN, and the next normal launch is exact again."""
    lens = [300, 257, 200, 190, 150, 140, 129, 100, 90, 80, 70, 65]
    p = workloads.prefill_inputs(lens, Heads(16, 16, 32), seed=22, gate="slow", state_scale=0.5)
    binding.prefill_giveups(reset=True)
    say("prefill persistent bounded waits: hooks off")
    o0, s0, a0 = _prefill_fault_injection(p, gpu, 0, 0)
    o1, s1 = run_prefill(p, gpu)
    torch.cuda.synchronize()
    assert int(a0.item()) == 0 and binding.prefill_giveups() == 0
    assert torch.equal(o0, o1) and torch.equal(s0, s1)
    say("prefill persistent bounded waits: chunk-ready signals stop after each chain's chunk 0")
    o2, s2, a2 = _prefill_fault_injection(p, gpu, 2000, 1)
    torch.cuda.synchronize()
    n = int(a2.item())
    cus = torch.cuda.get_device_properties(gpu).multi_processor_count
    assert cus < 12 * 32 and cus <= n <= cus * 8, (n, cus)
    assert binding.prefill_giveups(reset=True) == n, "the device counter must see every give-up"
    assert torch.isnan(o2.float()).all() and torch.isnan(s2).all()
    say("prefill persistent bounded waits: a normal launch afterwards")
    o3, s3 = run_prefill(p, gpu)
    torch.cuda.synchronize()
    assert torch.equal(o3, o1) and torch.equal(s3, s1)
    assert binding.prefill_giveups() == 0


@pytest.mark.parametrize("in_place", [False, True])
def test_prefill_dropin_scratch_path(gpu, in_place):
    """One sequence of at least 1,024 tokens through the drop-in runs two kernels in the
    library's drop-in scratch: a 2,500-token sequence with an initial state (updated in
    place or not) and int64 offsets against the oracle, twice in a row (the second call
    waits for the first one's use of the scratch), and bit for bit equal to
    gdn_prefill_with_workspace."""
    say(f"prefill drop-in scratch path, 2,500 tokens, in_place={in_place}")
    p = workloads.prefill_inputs([2500], seed=61, gate="slow", state_scale=0.5, cu_dtype=torch.int64)
    assert _dropin_windows(p) == (1, 0)
    o_ref, s_ref = oracle_prefill(p)
    out, ns = run_prefill(p, gpu, in_place=in_place)
    out2, ns2 = run_prefill(p, gpu, in_place=False)
    torch.cuda.synchronize()
    assert_close(host(out), o_ref, OUT_RTOL, OUT_ATOL, "output")
    assert_close(host(ns), s_ref, STATE_RTOL, STATE_ATOL, "new_state")
    assert torch.equal(out2, out)
    if not in_place:
        assert torch.equal(ns2, ns)
    o3, s3 = _prefill_capi(p, gpu, workspace=True)
    torch.cuda.synchronize()
    assert torch.equal(o3, out) and (in_place or torch.equal(s3, ns))


def test_prefill_dropin_long_sequence(gpu):
    """A 12,288-token sequence (32 v-heads: 118 MB of chunk images, most of the drop-in's
    scratch) runs two kernels there in one window: against the oracle, and bit for bit equal
    to gdn_prefill_with_workspace."""
    say("prefill drop-in, one 12,288-token sequence")
    lib = _lib.load()
    p = workloads.prefill_inputs([12288], seed=62, gate="slow", state_scale=0.5)
    need = lib.gdn_prefill_workspace_size(1, 12288, 32)
    assert 64 << 20 < need <= _lib.GDN_PREFILL_DROPIN_SCRATCH_BYTES, need
    assert _dropin_windows(p) == (1, 0)
    o_ref, s_ref = oracle_prefill(p)
    out, ns = run_prefill(p, gpu)
    o2, s2 = _prefill_capi(p, gpu, workspace=True)
    torch.cuda.synchronize()
    assert_close(host(out), o_ref, OUT_RTOL, OUT_ATOL, "output")
    assert_close(host(ns), s_ref, STATE_RTOL, STATE_ATOL, "new_state")
    assert torch.equal(out, o2) and torch.equal(ns, s2)


@pytest.mark.parametrize("lens,heads,windows,state,cu_dtype", [
    ([15001], Heads(16, 16, 32), 2, "in place", torch.int32),        # 32 chains, split 8 ways
    ([10500, 4700], Heads(16, 16, 32), 3, "new", torch.int64),       # 64 chains split 4 ways; one ends first
    ([28001], Heads(16, 16, 32), 3, None, torch.int32),              # no initial state
    ([19001], Heads(12, 12, 24), 2, "new", torch.int64),             # 192 workgroups
    ([0, 15000], Heads(16, 16, 32), 3, None, torch.int64),           # an empty sequence, zeroed once
    ([9400, 0], Heads(24, 24, 24), 1, "in place", torch.int32),      # split 4 ways, only as offsets that overlap
                                                                     # cannot come from two sequences
    ([3000, 5900], Heads(16, 16, 48), 1, "new", torch.int64),        # split 2 ways, the same
    ([8192, 8192], Heads(16, 16, 48), 0, "new", torch.int32),        # split 2 ways, beyond one window
    ([30000], Heads(8, 8, 16), 0, None, torch.int32),                # windows would leave half the CUs idle
])
def test_prefill_dropin_windows(gpu, lens, heads, windows, state, cu_dtype):
    """Batches whose chunk images exceed the drop-in's scratch run in windows of the
    sequences, the state carried from one to the next in new_state: the expected number of
    windows, within tolerance of the oracle, and bit for bit one kernel (and, where the batch
    takes a workspace, gdn_prefill_with_workspace, one window)."""
    say(f"prefill drop-in in windows, lens={lens} heads={heads} state={state}")
    lib = _lib.load()
    T, N = sum(lens), len(lens)
    assert N * ((T + 63) // 64) * heads.hv * 19200 > _lib.GDN_PREFILL_DROPIN_SCRATCH_BYTES
    p = workloads.prefill_inputs(lens, heads, seed=64, gate="slow", state_scale=0.5, with_state=state is not None,
                                 cu_dtype=cu_dtype)
    assert _dropin_windows(p) == (windows, int(windows > 0 and heads.hv * N > 64))
    o1, s1, aborts = _prefill_fault_injection(p, gpu, 0, 0)
    o_ref, s_ref = oracle_prefill(p)
    out, ns = run_prefill(p, gpu, in_place=state == "in place")
    torch.cuda.synchronize()
    assert int(aborts.item()) == 0
    assert torch.equal(out, o1) and torch.equal(ns, s1)
    if lib.gdn_prefill_workspace_size(N, T, heads.hv) > 0:
        o2, s2 = _prefill_capi(p, gpu, workspace=True)
        assert torch.equal(out, o2) and torch.equal(ns, s2)
    assert_close(host(out), o_ref, OUT_RTOL, OUT_ATOL, "output")
    assert_close(host(ns), s_ref, STATE_RTOL, STATE_ATOL, "new_state")


@pytest.mark.parametrize("lens,heads,two_kernels", [
    ([100, 2999, 900], Heads(16, 16, 32), True),     # 96 chains, split 2 ways
    ([1100, 64, 2000, 1], Heads(12, 6, 24), False),  # the same, below the average length
    ([1024, 1025, 1023], Heads(8, 16, 32), True),    # at the threshold, distinct head ratios
    ([700, 630], Heads(8, 8, 16), True),             # split 8 ways, above 640 tokens
    ([640], Heads(16, 16, 32), True),                # at it
    ([639], Heads(16, 16, 32), False),
])
def test_prefill_dropin_rule_edges(gpu, lens, heads, two_kernels):
    """Around the lines of the drop-in's choice between one kernel and two: the expected side
    of the line, bit for bit the one kernel (launched through the testing entry point with its
    hooks off), and within tolerance of the oracle."""
    say(f"prefill drop-in rule lens={lens} heads={heads} two_kernels={two_kernels}")
    p = workloads.prefill_inputs(lens, heads, seed=65, gate="slow", state_scale=0.5)
    assert _dropin_windows(p)[0] == int(two_kernels)
    o1, s1, aborts = _prefill_fault_injection(p, gpu, 0, 0)
    o2, s2 = run_prefill(p, gpu)
    torch.cuda.synchronize()
    assert int(aborts.item()) == 0
    assert torch.equal(o1, o2) and torch.equal(s1, s2)
    o_ref, s_ref = oracle_prefill(p)
    assert_close(host(o2), o_ref, OUT_RTOL, OUT_ATOL, "output")
    assert_close(host(s2), s_ref, STATE_RTOL, STATE_ATOL, "new_state")
