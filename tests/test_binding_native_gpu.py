"""The native call path of the Python entry points (gdn_kernel_amd._native): it launches the
calls it matches with the results of the Python path, and leaves every other call, in all
the forms the Python path takes or refuses, to it."""
import pytest
import torch

from gdn_kernel_amd import _lib, binding, workloads
from tests.gpu_util import say

pytestmark = pytest.mark.gpu


class _Counting:
    """The native module, counting the calls it took."""

    def __init__(self, mod):
        self.mod, self.taken = mod, 0

    def __getattr__(self, name):
        def call(*args):
            rc = getattr(self.mod, name)(*args)
            self.taken += rc is not None
            return rc
        return call


@pytest.fixture
def native(gpu, monkeypatch):
    mod = _lib.native()
    assert hasattr(mod, "bind"), "the native module is not built"
    counting = _Counting(mod)
    monkeypatch.setattr(_lib, "_native", counting)
    return counting


def _run(native, monkeypatch, call, expect_taken):
    """`call` with and without the native module; the outputs of both."""
    native.taken = 0
    with_native = call()
    assert (native.taken == 1) == expect_taken
    with monkeypatch.context() as m:
        m.setattr(_lib, "_native", _lib._NoNative)
        python = call()
    torch.cuda.synchronize()
    for x, y in zip(with_native, python):
        assert torch.equal(x, y)


@pytest.mark.parametrize("form", ["plain", "null_state", "default_scale", "int_scale", "parameter", "subclass"])
def test_decode_forms(native, gpu, monkeypatch, form):
    say(f"native decode, {form}")
    w = workloads.decode_inputs(3, seed=5, device=gpu, gate="slow", state_scale=0.5)
    scale = {"default_scale": None, "int_scale": 1}.get(form, w["scale"])
    q = w["q"]
    if form == "parameter":
        q = torch.nn.Parameter(q, requires_grad=False)
    elif form == "subclass":
        q = q.as_subclass(type("Sub", (torch.Tensor,), {}))

    def call():
        out, ns = torch.empty_like(w["v"]), torch.empty_like(w["state"])
        binding.decode_kernel(q, w["k"], w["v"], None if form == "null_state" else w["state"], w["A_log"], w["a"],
                              w["dt_bias"], w["b"], scale, out, ns)
        return out, ns

    _run(native, monkeypatch, call, form not in ("int_scale", "subclass"))


def test_pooled(native, gpu, monkeypatch):
    say("native pooled decode")
    w = workloads.decode_inputs(5, seed=6, device=gpu, gate="slow", state_scale=0.5, pool_slots=9)
    w["state_indices"][2] = -1

    def call():
        out, pool = torch.empty_like(w["v"]), w["state"].clone()
        binding.decode_pooled_kernel(w["q"], w["k"], w["v"], pool, w["A_log"], w["a"], w["dt_bias"], w["b"],
                                     w["scale"], out, w["state_indices"])
        return out, pool

    _run(native, monkeypatch, call, True)


@pytest.mark.parametrize("form", ["int32", "int64", "null_state", "leading_one", "workspace"])
def test_prefill_forms(native, gpu, monkeypatch, form):
    say(f"native prefill, {form}")
    p = workloads.prefill_inputs([70, 0, 9], seed=7, device=gpu, gate="slow", state_scale=0.5,
                                 cu_dtype=torch.int64 if form == "int64" else torch.int32)
    n = binding.prefill_workspace_bytes(3, 79, 32)
    lead = (lambda t: t[None]) if form == "leading_one" else (lambda t: t)

    def call():
        out, ns = torch.empty_like(p["v"]), torch.empty_like(p["state"])
        args = [lead(p["q"]), lead(p["k"]), lead(p["v"]), None if form == "null_state" else p["state"], p["A_log"],
                lead(p["a"]), p["dt_bias"], lead(p["b"]), p["cu_seqlens"], p["scale"], lead(out), ns]
        if form == "workspace":
            binding.prefill_kernel_with_workspace(*args, torch.empty(max(n, 16), dtype=torch.uint8, device=gpu))
        else:
            binding.prefill_kernel(*args)
        return out, ns

    _run(native, monkeypatch, call, form != "leading_one")


@pytest.mark.parametrize("bad,match", [
    (dict(q=lambda t: t.float()), "q must be torch.bfloat16"),
    (dict(k=lambda t: torch.cat([t, t], -1)[..., :128]), "k must be contiguous"),
    (dict(state=lambda t: t[:1]), "state must have shape"),
    (dict(v=lambda t: t.cpu()), "v is on cpu"),
    (dict(a=lambda t: None), "a must be a torch.Tensor"),
    (dict(q=lambda t: t.view(2, 16, 128)), "4-D"),
    (dict(scale=lambda s: float("inf")), "scale must be finite"),
    (dict(new_state=lambda t: t[:, :31].contiguous()), "new_state must have shape"),
])
def test_refusals_keep_their_messages(native, gpu, bad, match):
    say(f"native refusal: {match}")
    w = workloads.decode_inputs(2, seed=8, device=gpu)
    w.update(output=torch.empty_like(w["v"]), new_state=torch.empty_like(w["state"]))
    for name, change in bad.items():
        w[name] = change(w[name])
    with pytest.raises(ValueError, match=match):
        binding.decode_kernel(*(w[n] for n in ("q", "k", "v", "state", "A_log", "a", "dt_bias", "b", "scale",
                                               "output", "new_state")))
