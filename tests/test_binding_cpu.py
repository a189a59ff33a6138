"""CPU tests of the Python binding's argument checks and of the workload
generators (no GPU; nothing is launched)."""
import math
import struct
import sys

import numpy as np
import pytest
import torch

from gdn_kernel_amd import _lib, binding, workloads


@pytest.mark.parametrize("missing", ["library", "unloadable library", "GPU build of torch"])
def test_arguments_are_checked_before_the_library(monkeypatch, tmp_path, missing):
    """Bad arguments are reported as such where the library or torch's GPU functions are
    missing; with the library missing, a call that passes its checks raises ImportError."""
    monkeypatch.setattr(_lib, "_native", None)
    if missing == "GPU build of torch":
        monkeypatch.delattr(torch._C, "_cuda_getDevice")
    else:
        monkeypatch.setattr(_lib, "_lib", None)
        monkeypatch.setattr(_lib, "LIB_PATH", tmp_path / "absent.so")
        if missing == "unloadable library":
            (tmp_path / "absent.so").write_bytes(b"not a library")
    w = workloads.decode_inputs(2, seed=0, pool_slots=3)
    p = workloads.prefill_inputs([3, 5], seed=0)
    decode = [w[n] for n in ("q", "k", "v", "state", "A_log", "a", "dt_bias", "b", "scale")] + [w["v"]]
    prefill = [p[n] for n in ("q", "k", "v", "state", "A_log", "a", "dt_bias", "b", "cu_seqlens", "scale")]
    prefill += [p["v"], p["state"]]
    for call in (lambda: binding.decode_kernel(*decode, w["state"]),
                 lambda: binding.decode_pooled_kernel(*decode, w["state_indices"]),
                 lambda: binding.prefill_kernel(*prefill),
                 lambda: binding.prefill_kernel_with_workspace(*prefill, None)):
        with pytest.raises(ValueError, match="GPU"):
            call()
    if missing == "library":
        with pytest.raises(ImportError, match="not built"):
            _lib.load()


class _Module:
    """A stand-in for the built native module."""

    def __init__(self, **stamps):
        self.bound = False
        self.__dict__.update(stamps)

    def bind(self, *args):
        self.bound = True


def _native_with(monkeypatch, module):
    """_lib.native() where `module` (None: no file; an exception: its import raises it) is
    the package's native module."""
    monkeypatch.setattr(_lib, "_native", None)
    spec = None if module is None else object()
    monkeypatch.setattr(_lib.importlib.util, "find_spec", lambda name: spec)
    package = sys.modules["gdn_kernel_amd"]
    monkeypatch.delattr(package, "_native", raising=False)
    monkeypatch.delitem(sys.modules, "gdn_kernel_amd._native", raising=False)
    if isinstance(module, Exception):
        class Finder:
            @staticmethod
            def find_spec(name, path=None, target=None):
                if name == "gdn_kernel_amd._native":
                    raise module
        monkeypatch.setattr(sys, "meta_path", [Finder, *sys.meta_path])
    elif module is not None:
        monkeypatch.setattr(package, "_native", module, raising=False)
    return _lib.native()


def test_native_module_that_does_not_match_is_refused(monkeypatch):
    """Only a missing native module leaves the calls to the Python code: one that does not
    load, or that was built for another torch or another library (or before it was
    stamped), raises."""
    torch_version, library = str(torch.__version__), _lib.load().gdn_build_id().decode()
    good = _Module(torch_version=torch_version, library_build_id=library)
    assert _native_with(monkeypatch, good) is good and good.bound
    assert _native_with(monkeypatch, None) is _lib._NoNative
    with pytest.raises(ImportError, match="does not load"):
        _native_with(monkeypatch, ImportError("undefined symbol"))
    for stamps, what in (({}, "torch"), (dict(torch_version="1.0", library_build_id=library), "torch"),
                         (dict(torch_version=torch_version, library_build_id="0" * 16), "library"),
                         (dict(torch_version=torch_version), "library")):
        with pytest.raises(ImportError, match=f"another version of .*{what}"):
            _native_with(monkeypatch, _Module(**stamps))


def test_native_module_is_built_from_these_sources():
    from gdn_kernel_amd import _native, build
    assert _native.build_id == build.native_digest()
    assert _native.library_build_id == build.source_digest() == _lib.load().gdn_build_id().decode()
    assert _native.torch_version == str(torch.__version__)


def test_native_module_has_no_tls_segment():
    """A TLS segment in the module would slow down every torch call of the thread that
    imports it (see build_native)."""
    from gdn_kernel_amd import build
    elf = build.native_path().read_bytes()
    assert elf[:6] == b"\x7fELF\x02\x01"
    at, size, count = (struct.unpack_from("<Q", elf, 0x20)[0], *struct.unpack_from("<HH", elf, 0x36))
    types = [struct.unpack_from("<I", elf, at + i * size)[0] for i in range(count)]
    assert 1 in types and 7 not in types            # PT_LOAD, no PT_TLS


@pytest.mark.parametrize("cxx", ["absent", "failing"])
def test_build_without_a_host_compiler(monkeypatch, tmp_path, capsys, cxx):
    """Without a working host compiler `python -m gdn_kernel_amd.build` still builds the
    library and goes on to the TVM-FFI shims; a native module of an earlier build, which
    would not match, goes."""
    from gdn_kernel_amd import build
    compiler = tmp_path / "c++"
    if cxx == "failing":
        compiler.write_text("#!/bin/sh\nexit 1\n")
        compiler.chmod(0o755)
    monkeypatch.setenv("CXX", str(compiler))
    (tmp_path / "_native.so").write_bytes(b"")
    shims = []
    monkeypatch.setattr(build, "build", lambda verbose: tmp_path / "lib.so")
    monkeypatch.setattr(build, "native_path", lambda: tmp_path / "_native.so")
    monkeypatch.setattr(build, "build_tvm_ffi", lambda verbose: shims.append(1) or {})
    build.main()
    out = capsys.readouterr().out
    assert "lib.so" in out and "native module not built" in out and shims == [1]
    assert not (tmp_path / "_native.so").exists()


def test_binding_rejects_cpu_tensors():
    w = workloads.decode_inputs(2, seed=0)
    out = torch.empty_like(w["v"])
    with pytest.raises(ValueError, match="GPU"):
        binding.decode_kernel(w["q"], w["k"], w["v"], w["state"], w["A_log"], w["a"],
                              w["dt_bias"], w["b"], w["scale"], out, w["state"])
    p = workloads.prefill_inputs([3, 5], seed=0)
    with pytest.raises(ValueError, match="GPU"):
        binding.prefill_kernel(p["q"], p["k"], p["v"], p["state"], p["A_log"], p["a"],
                               p["dt_bias"], p["b"], p["cu_seqlens"], p["scale"],
                               torch.empty_like(p["v"]), torch.empty_like(p["state"]))


def test_prefill_with_workspace_checks_arguments():
    p = workloads.prefill_inputs([3, 5], seed=0)
    with pytest.raises(ValueError, match="GPU"):
        binding.prefill_kernel_with_workspace(
            p["q"], p["k"], p["v"], p["state"], p["A_log"], p["a"], p["dt_bias"], p["b"],
            p["cu_seqlens"], p["scale"], torch.empty_like(p["v"]), torch.empty_like(p["state"]),
            torch.empty(16, dtype=torch.uint8))


def test_entry_points_have_reference_arity():
    import inspect
    from gdn_kernel_amd import decode, prefill
    assert list(inspect.signature(decode.kernel).parameters) == [
        "q", "k", "v", "state", "A_log", "a", "dt_bias", "b", "scale", "output", "new_state"]
    assert list(inspect.signature(prefill.kernel).parameters) == [
        "q", "k", "v", "state", "A_log", "a", "dt_bias", "b", "cu_seqlens", "scale", "output",
        "new_state"]


def test_decode_inputs_distribution():
    w = workloads.decode_inputs(64, seed=1)
    assert w["q"].dtype == torch.bfloat16 and w["q"].shape == (64, 1, 16, 128)
    n = w["q"].float().norm(dim=-1)
    assert torch.allclose(n, torch.ones_like(n), atol=1e-2)
    A = torch.exp(w["A_log"])
    assert (A >= 1).all() and (A <= 16).all()
    assert w["state"].shape == (64, 32, 128, 128)
    assert abs(float(w["state"].std()) - 0.05) < 1e-3
    assert w["scale"] == 1 / math.sqrt(128)


def test_pool_indices_are_distinct_permutation():
    w = workloads.decode_inputs(512, seed=2, pool_slots=1024)
    idx = w["state_indices"]
    assert idx.dtype == torch.int32 and idx.shape == (512,)
    assert len(set(idx.tolist())) == 512 and int(idx.min()) >= 0 and int(idx.max()) < 1024


def test_varlen_lengths():
    lens = workloads.varlen_lengths(32, 32768)
    assert len(lens) == 32 and sum(lens) == 32768
    assert min(lens) >= 1 and min(lens) < 64 and max(lens) >= 4096 // 2
    assert lens == workloads.varlen_lengths(32, 32768)          # deterministic


def test_prefill_inputs_layout():
    p = workloads.prefill_inputs([5, 0, 70], seed=3, cu_dtype=torch.int64)
    assert p["q"].shape == (75, 16, 128) and p["v"].shape == (75, 32, 128)
    assert p["cu_seqlens"].tolist() == [0, 5, 5, 75] and p["cu_seqlens"].dtype == torch.int64
    assert p["state"].shape == (3, 32, 128, 128)


def test_to_numpy_exact():
    x = torch.randn(100).to(torch.bfloat16)
    y = workloads.to_numpy(x)
    assert y.dtype == np.float64 and np.array_equal(y, x.float().numpy().astype(np.float64))
