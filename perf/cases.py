"""Workloads of this library as its users run them, for timing and comparing builds.

A case is a plain dict: the operation ("decode", "pooled" or "prefill"), its sizes and
options.  Head layouts are 16 q / 16 k / 32 v heads (a whole layer on one GPU) and its
tensor-parallel shares 8 / 8 / 16 and 4 / 4 / 8, all with 128 columns a head.  Inputs come
from ``gdn_kernel_amd.workloads`` (normalised bf16 q and k, bf16 v, a and b, fp32 states
and parameters), outputs are preallocated as the destination-passing entry points take
them, and the state is updated in place where a serving program does so.
"""
import math

import torch

from gdn_kernel_amd import binding, workloads
from gdn_kernel_amd.decode import kernel as decode
from gdn_kernel_amd.prefill import kernel as prefill

D = 128
HEADS = ((16, 16, 32), (8, 8, 16), (4, 4, 8))
MAX_TOKENS = 32768                   # of a packed batch
MAX_LENGTH = 16384                   # of one sequence
CHUNK_FLOP = 180224                  # per token and v-head, chunks of 64: 2 (5 * 64 * 128 + 3 * 128 * 128)


def _decode(name, batch, heads=HEADS[0], gate="baseline"):
    return {"name": name, "op": "decode", "batch": batch, "hq": heads[0], "hk": heads[1], "hv": heads[2],
            "gate": gate}


def _pooled(name, batch, slots, padding=0, heads=HEADS[0], gate="baseline"):
    return {"name": name, "op": "pooled", "batch": batch, "slots": slots, "padding": padding,
            "hq": heads[0], "hk": heads[1], "hv": heads[2], "gate": gate}


def _prefill(name, lengths, heads=HEADS[0], gate="baseline", state=True, in_place=False, cu64=False,
             workspace=False):
    return {"name": name, "op": "prefill", "lengths": ",".join(str(int(x)) for x in lengths),
            "hq": heads[0], "hk": heads[1], "hv": heads[2], "gate": gate, "state": state,
            "in_place": in_place, "cu64": cu64, "workspace": workspace}


def listed():
    return [
        # One user's token: the smallest call, all launch and latency.
        _decode("decode_b1", 1),
        # A small odd batch on one of four tensor-parallel GPUs.
        _decode("decode_b13_tp4", 13, HEADS[2]),
        # The headline step: a full batch updating its state in place.
        _decode("decode_b64", 64),
        # A serving engine's ragged step over its slot pool: fixed launch size, some rows unused.
        _pooled("pooled_b24_padded", 24, 64, padding=5),
        # A large serving step over a large pool.
        _pooled("pooled_b512", 512, 1024),
        # A short chat prompt, no state yet: less than one chunk.
        _prefill("prefill_37", [37], state=False),
        # The next slice of a prompt that is fed in slices, its state carried in place.
        _prefill("prefill_512_continued", [512], in_place=True, cu64=True),
        # One ordinary long prompt.
        _prefill("prefill_4096", [4096], state=False),
        # A whole document: the longest single sequence.
        _prefill("prefill_16384", [16384], state=False),
        # A few prompts of different lengths prefilled together.
        _prefill("prefill_4_ragged", [1000, 1500, 300, 1307]),
        # The headline varlen batch.
        _prefill("prefill_32_varlen_32k", workloads.varlen_lengths(workloads.CONFIG4_NUM_SEQS,
                                                                   workloads.CONFIG4_TOTAL)),
        # Many short prompts at once (an evaluation or classification run).
        _prefill("prefill_48_short", [1 + (37 * i * i + 11 * i) % 200 for i in range(48)]),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    heads = HEADS[rng.choice((0, 0, 0, 1, 2))]
    gate = rng.choice(("baseline", "baseline", "slow"))
    op = rng.choice(("decode", "pooled", "prefill", "prefill", "prefill"))
    if op == "decode":
        c = _decode("", _log_int(rng, 2, 256), heads, gate)
    elif op == "pooled":
        batch = _log_int(rng, 2, 512)
        c = _pooled("", batch, _log_int(rng, batch, 1024), rng.choice((0, 0, batch // 4)), heads, gate)
    else:
        seqs = _log_int(rng, 1, 64)
        total = _log_int(rng, max(16, seqs), MAX_TOKENS)
        share = [math.exp(rng.uniform(0.0, math.log(max(2.0, total / seqs)))) for _ in range(seqs)]
        lengths = [min(MAX_LENGTH, max(1, int(total * s / sum(share)))) for s in share]
        state = rng.random() < 0.7
        c = _prefill("", lengths, heads, gate, state, state and rng.random() < 0.5, rng.random() < 0.3,
                     rng.random() < 0.2)
    del c["name"]
    return c


def _heads(case):
    return workloads.Heads(case["hq"], case["hk"], case["hv"])


def _lengths(case):
    return [int(x) for x in case["lengths"].split(",")]


def _inputs(case, seed):
    """The inputs of `case`, on the GPU."""
    dev, heads, gate = torch.device("cuda", torch.cuda.current_device()), _heads(case), case["gate"]
    if case["op"] == "decode":
        return workloads.decode_inputs(case["batch"], heads, seed, dev, gate)
    if case["op"] == "pooled":
        p = workloads.decode_inputs(case["batch"], heads, seed, dev, gate, pool_slots=case["slots"])
        if case["padding"]:                       # unused rows of a fixed-size launch, anywhere in the batch
            gen = torch.Generator(device=dev)
            gen.manual_seed(seed + 1)
            p["state_indices"][torch.randperm(case["batch"], generator=gen, device=dev)[:case["padding"]]] = -1
        return p
    return workloads.prefill_inputs(_lengths(case), heads, seed, dev, gate, with_state=case["state"],
                                    cu_dtype=torch.int64 if case["cu64"] else torch.int32)


def prepare(case, seed):
    p = _inputs(case, seed)
    p["op"] = case["op"]
    p["out"] = torch.empty_like(p["v"])
    if case["op"] == "decode":
        p["new_state"] = p["state"]
    elif case["op"] == "prefill":
        n = len(p["lengths"])
        p["new_state"] = p["state"] if case["in_place"] else \
            torch.empty((n, case["hv"], D, D), dtype=torch.float32, device=p["v"].device)
        nbytes = binding.prefill_workspace_bytes(n, p["v"].shape[0], case["hv"]) if case["workspace"] else 0
        p["workspace"] = torch.empty(nbytes, dtype=torch.uint8, device=p["v"].device) if nbytes else None
    return p


def run(p):
    if p["op"] == "decode":
        decode(p["q"], p["k"], p["v"], p["state"], p["A_log"], p["a"], p["dt_bias"], p["b"], p["scale"],
               p["out"], p["new_state"])
        return p["out"], p["new_state"]
    if p["op"] == "pooled":
        binding.decode_pooled_kernel(p["q"], p["k"], p["v"], p["state"], p["A_log"], p["a"], p["dt_bias"], p["b"],
                                     p["scale"], p["out"], p["state_indices"])
        return p["out"], p["state"]
    args = (p["q"], p["k"], p["v"], p["state"], p["A_log"], p["a"], p["dt_bias"], p["b"], p["cu_seqlens"],
            p["scale"], p["out"], p["new_state"])
    if p["workspace"] is not None:
        binding.prefill_kernel_with_workspace(*args, p["workspace"])
    else:
        prefill(*args)
    return p["out"], p["new_state"]


def work(case):
    hq, hk, hv = case["hq"], case["hk"], case["hv"]
    token = 2 * D * (hq + hk + 2 * hv) + 2 * 2 * hv          # q, k, v, the output, a and b
    params = 2 * 4 * hv
    state = 4 * hv * D * D
    if case["op"] == "prefill":
        lengths = _lengths(case)
        n, t = len(lengths), sum(lengths)
        return {"bytes": token * t + params + state * n * (2 if case["state"] else 1),
                "flops": CHUNK_FLOP * hv * t}
    rows = case["batch"] - case.get("padding", 0)
    index = 4 * case["batch"] if case["op"] == "pooled" else 0
    # per state element: the decay, two dot products and the rank-1 update
    return {"bytes": token * rows + params + 2 * state * rows + index, "flops": 7 * D * D * hv * rows}


def tolerance(case):
    # The bf16 output: relative rms error against 64 bits 1.7e-3 (decode: its rounding) and
    # 2.9e-3 (prefill: products that only reach the output have bf16 operands) as measured;
    # the fp32 state: 1e-7 and 3e-6.  "max" is against the root mean square.
    return {"rel": 1e-2, "max": 8e-2}


def _gates(p, rows):
    """(log decay, beta) in 64 bits, [rows, Hv]."""
    x = p["a"].double().view(rows, -1) + p["dt_bias"].double()
    return -torch.exp(p["A_log"].double()) * torch.nn.functional.softplus(x), \
        torch.sigmoid(p["b"].double().view(rows, -1))


def _per_v_head(x, hv):
    return x.double().repeat_interleave(hv // x.shape[-2], dim=-2)


def _exact_decode(p, hv, state):
    """(output [B, Hv, D], new state) in 64 bits for rows whose states are `state`."""
    q, k, v = (_per_v_head(p[n][:, 0], hv) for n in ("q", "k", "v"))
    log_g, beta = _gates(p, q.shape[0])
    s = state.double() * torch.exp(log_g)[..., None, None]
    delta = beta[..., None] * (v - (s @ k[..., None])[..., 0])
    s += delta[..., None] * k[..., None, :]
    return p["scale"] * (s @ q[..., None])[..., 0], s


def _exact_prefill(p, hv, lengths):
    """The chunked form of the recurrence in 64 bits, one sequence after another."""
    t = p["v"].shape[0]
    dev = p["v"].device
    q, k, v = (_per_v_head(p[n], hv).transpose(0, 1) for n in ("q", "k", "v"))     # [Hv, T, D]
    log_g, beta = (x.t() for x in _gates(p, t))                                    # [Hv, T]
    out = torch.empty((hv, t, D), dtype=torch.float64, device=dev)
    states = []
    at = 0
    for i, n in enumerate(lengths):
        s = p["state"][i].double() if p["state"] is not None else \
            torch.zeros((hv, D, D), dtype=torch.float64, device=dev)
        for c0 in range(at, at + n, 64):
            c = slice(c0, min(c0 + 64, at + n))
            m = c.stop - c.start
            kc, qc, gam, bet = k[:, c], q[:, c], torch.cumsum(log_g[:, c], 1), beta[:, c, None]
            low = torch.ones((m, m), dtype=torch.bool, device=dev).tril()
            decay = torch.exp((gam[:, :, None] - gam[:, None, :]).masked_fill(~low, -math.inf))
            eye = torch.eye(m, dtype=torch.float64, device=dev)
            lhs = eye + (bet * decay * (kc @ kc.transpose(1, 2))).tril(-1)
            rhs = bet * (v[:, c] - torch.exp(gam)[..., None] * (kc @ s.transpose(1, 2)))
            u = torch.linalg.solve_triangular(lhs, rhs, upper=False, unitriangular=True)
            out[:, c] = p["scale"] * (torch.exp(gam)[..., None] * (qc @ s.transpose(1, 2)) +
                                      (decay * (qc @ kc.transpose(1, 2))) @ u)
            last = gam[:, -1:]
            s = torch.exp(last)[..., None] * s + \
                (torch.exp(last - gam)[..., None] * u).transpose(1, 2) @ kc
        states.append(s)
        at += n
    return out.transpose(0, 1), torch.stack(states)


def exact(case, seed):
    p = _inputs(case, seed)
    hv = case["hv"]
    if case["op"] == "decode":
        o, s = _exact_decode(p, hv, p["state"])
        return o[:, None], s
    if case["op"] == "pooled":
        rows = (p["state_indices"] >= 0).nonzero()[:, 0]
        slots = p["state_indices"][rows].long()
        live = {n: (x[rows] if n in ("q", "k", "v", "a", "b") else x) for n, x in p.items()}
        o, s = _exact_decode(live, hv, p["state"][slots])
        out = torch.zeros((case["batch"], 1, hv, D), dtype=torch.float64, device=o.device)
        out[rows, 0] = o
        pool = p["state"].double()
        pool[slots] = s
        return out, pool
    return _exact_prefill(p, hv, _lengths(case))
