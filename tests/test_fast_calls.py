"""The C++ host side of the eager calls leaves to the Python code whatever is not a plain ROCm tensor.

Runs without a GPU: every form here must come back as None (nothing called),
and the public calls must raise what they raised before.
"""

from __future__ import annotations

import warnings

import pytest
import torch

from liteinfer_amd import _native
from liteinfer_amd.paged_kernels import paged_decode
from liteinfer_amd.rope import rope_kv_write

pytestmark = pytest.mark.skipif(not _native.is_built(), reason="the HIP library is not built")


def _operands():
    q, pool = torch.zeros(2, 8, 64, dtype=torch.bfloat16), torch.zeros(32, 2, 64, dtype=torch.bfloat16)
    return [q, pool, pool.clone(), torch.zeros(2, 5, dtype=torch.int64), torch.ones(2, dtype=torch.int32)]


class _Sub(torch.Tensor):
    pass


@pytest.mark.parametrize("swap", [lambda t: t, lambda t: t.as_subclass(_Sub), lambda t: t.to("meta"), lambda t: None,
                                  lambda t: t.tolist()])
def test_left_to_python(swap):
    f = _native.fast_calls()
    ops = [swap(t) for t in _operands()]
    assert f.decode(*ops, 0.125, 4, 64, 0, 0, 1.0, 1.0, None, None, 0) is None
    assert f.rope(*(swap(torch.zeros(1, 2, 3, 64)) for _ in range(3)), *ops, 1.0, 1.0, None, 0) is None
    assert f.prefill(*ops, ops[4], 1, 0.125, 4, 32, 16, 0, 1.0, 1.0, None, 0) is None
    assert f.decode(*ops) is None and f.prefill() is None and f.rope() is None  # too few arguments


def test_the_calls_still_raise():
    with pytest.raises(RuntimeError, match="need a ROCm device"):
        paged_decode(*_operands(), 0.125, 4)
    with pytest.raises(ValueError, match="num_splits must be >= 1"):
        paged_decode(*_operands(), 0.125, 4, num_splits=0)
    x = torch.zeros(1, 2, 3, 64)
    with pytest.raises(RuntimeError, match="need a ROCm device"):
        rope_kv_write(x, x, x, x[0], x[0], torch.zeros(3, dtype=torch.int64), x[0], x[0])


def test_a_module_of_other_sources_is_refused(monkeypatch):
    monkeypatch.setattr(_native, "_fast", None)
    monkeypatch.setattr(_native._build, "source_hash", lambda: "0" * 16)
    monkeypatch.setattr(_native, "load", lambda: object())
    with pytest.raises(RuntimeError, match="built from other sources"):
        _native.fast_calls()


@pytest.mark.parametrize("owner,name,value", [
    (torch, "__version__", "9.9.9"), (torch.version, "git_version", "f" * 40),
    (torch._C, "_GLIBCXX_USE_CXX11_ABI", not torch._C._GLIBCXX_USE_CXX11_ABI),
    (_native._build.sys.implementation, "cache_tag", "cpython-99"), (_native._build, "FAST_CALLS_FLAGS", ["-O3"]),
])
def test_a_module_for_another_torch_or_interpreter_is_not_found(monkeypatch, owner, name, value):
    built = _native._build.fast_calls_path()
    assert built.exists()
    monkeypatch.setattr(owner, name, value)
    assert not _native._build.fast_calls_path().exists()
    monkeypatch.undo()
    assert _native._build.fast_calls_path() == built


def _cannot_load(path):
    raise ImportError("undefined symbol")


@pytest.mark.parametrize("break_it", [
    lambda m, tmp: m.setattr(_native._build, "LIB_DIR", tmp),  # not there
    lambda m, tmp: m.setattr(_native, "_load_fast_calls", _cannot_load),
])
def test_without_the_module_the_python_code_serves_every_call(monkeypatch, tmp_path, break_it):
    monkeypatch.setattr(_native, "_fast", None)
    break_it(monkeypatch, tmp_path)
    with pytest.warns(RuntimeWarning, match="run through Python"):
        f = _native.fast_calls()
    assert f.decode(*_operands(), 0.125, 4) is None and f.prefill() is None and f.rope(1) is None
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        assert _native.fast_calls() is f  # (said once)


def test_a_failed_extension_build_does_not_end_the_build(monkeypatch, tmp_path, capsys):
    build = _native._build
    monkeypatch.setattr(build, "LIB_DIR", tmp_path)
    monkeypatch.setattr(build, "LIB_PATH", tmp_path / "lib.so")
    monkeypatch.setattr(build, "FAST_CALLS_FLAGS", ["--no-such-flag"])
    monkeypatch.setattr(build, "sources", lambda: [build.CSRC_DIR / "kv_scatter.hip"])
    (tmp_path / "_fast_calls.0.so").touch()
    assert build.build().exists()
    assert "will run through Python" in capsys.readouterr().err
    assert not list(tmp_path.glob("_fast_calls*"))
