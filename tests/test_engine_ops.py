"""What the engine's ops (engine/ops.py) do with operands their kernels do not serve (CPU; no kernel runs).

The kernels take raw pointers: a mismatched operand must be left to torch or
refused before one is handed over. `_OnGpu` stands for a tensor on a ROCm
device, and every launch fails the test.
"""

from __future__ import annotations

from types import SimpleNamespace

import pytest
import torch
import torch.nn.functional as F

from liteinfer_amd.engine import ops
from liteinfer_amd.engine.model import RandomLlama
from liteinfer_amd.engine.runner import DecodeGraphs


class _OnGpu(torch.Tensor):
    is_cuda = True
    device = torch.device("cuda", 0)


class _OnOther(_OnGpu):
    device = torch.device("cuda", 1)


def _gpu(*shape, dtype=torch.bfloat16, cls=_OnGpu):
    return torch.zeros(*shape, dtype=dtype).as_subclass(cls)


@pytest.fixture(autouse=True)
def no_launch(monkeypatch):
    class NoLibrary:
        def __getattr__(self, name):
            pytest.fail(f"{name} was called")

    monkeypatch.setattr(ops, "_splits", lambda rows, n, k: 1)
    monkeypatch.setattr(ops._native, "load", NoLibrary)


@pytest.mark.parametrize("op", [ops.linear, ops.linear_sums])
def test_projections_of_host_tensors_are_torchs(op):
    x, w = torch.randn(4, 256).to(torch.bfloat16), torch.randn(16, 256).to(torch.bfloat16)
    assert torch.equal(op(x, w), F.linear(x, w))
    with pytest.raises(RuntimeError, match="shapes cannot be multiplied"):
        op(x[:, :128], w)


@pytest.mark.parametrize("x,w", [
    (_gpu(4, 2048), _gpu(16, 4096)),  # a K of another length: past x's rows
    (_gpu(4, 4096), _gpu(16, 2048)),
    (_gpu(4, 256), torch.zeros(16, 256, dtype=torch.bfloat16)),  # a host weight
    (torch.zeros(4, 256, dtype=torch.bfloat16), _gpu(16, 256)),
    (_gpu(4, 256), _gpu(16, 256, cls=_OnOther)),
    (_gpu(4, 256), _gpu(256)),
    (_gpu(4, 256), _gpu(2, 8, 256)),
    (_gpu(4, 256), _gpu(16, 256, dtype=torch.float16)),
    (_gpu(4, 256).requires_grad_(), _gpu(16, 256)),  # the kernels record no graph
    (_gpu(4, 256), _gpu(16, 256).requires_grad_()),
])
def test_operands_that_do_not_fit_are_left_to_torch(x, w):
    assert ops._skinny(x, w)[1] == 0


def test_operands_that_fit_are_served():
    for x in (_gpu(4, 256), _gpu(2, 2, 256), _gpu(256), _gpu(1, 256).expand(4, 256)):
        assert ops._skinny(x, _gpu(16, 256))[1] == 1
    with torch.no_grad():
        assert ops._skinny(_gpu(4, 256), _gpu(16, 256).requires_grad_())[1] == 1


def test_an_empty_projection_is_torchs(monkeypatch):
    monkeypatch.undo()  # the rule itself
    assert ops._splits(4, 0, 256) == 0 and ops._splits(4, 16, 0) == 0


def test_host_tensors_are_refused():
    x, weight = torch.zeros(4, 256, dtype=torch.bfloat16), torch.ones(256, dtype=torch.bfloat16)
    with pytest.raises(ValueError, match="one ROCm device"):
        ops.gate_up_silu(x, torch.zeros(32, 256, dtype=torch.bfloat16))
    with pytest.raises(ValueError, match="one ROCm device"):
        ops.silu_mul(x)
    with pytest.raises(ValueError, match="one ROCm device"):
        ops.add_rms_norm(x, weight, 1e-5)
    with pytest.raises(ValueError, match="one ROCm device"):
        ops.add_rms_norm(_gpu(4, 256), weight, 1e-5)
    with pytest.raises(ValueError, match="one ROCm device"):
        ops.rotary_tables(torch.zeros(1, 3, dtype=torch.int64), torch.ones(32), torch.bfloat16)


@pytest.mark.parametrize("sums", [
    _gpu(2, 4, 256, dtype=torch.bfloat16), _gpu(2, 3, 256, dtype=torch.float32), _gpu(2, 4, 128, dtype=torch.float32),
    _gpu(4, 256, dtype=torch.float32), _gpu(2, 4, 512, dtype=torch.float32)[:, :, :256],
    torch.zeros(2, 4, 256), _gpu(2, 4, 256, dtype=torch.float32, cls=_OnOther)])
def test_sums_that_are_not_the_rows_are_refused(sums):
    with pytest.raises(ValueError):
        ops.add_rms_norm(_gpu(4, 256), _gpu(256), 1e-5, ops.Partials(sums, torch.Size((4, 256))))


@pytest.mark.parametrize("positions,inv_freq", [
    (_gpu(1, 3, dtype=torch.int64), torch.ones(32)),
    (torch.zeros(1, 3, dtype=torch.int64), _gpu(32, dtype=torch.float32)),
    (_gpu(1, 3, dtype=torch.float32), _gpu(32, dtype=torch.float32)),
    (_gpu(1, 3, dtype=torch.int64), _gpu(32, dtype=torch.float64)),
    (_gpu(1, 3, dtype=torch.int64), _gpu(64, dtype=torch.float32)[::2]),
    (_gpu(1, 3, dtype=torch.int64), _gpu(4, 8, dtype=torch.float32)),
])
def test_rotary_operands_are_checked(positions, inv_freq):
    with pytest.raises(ValueError):
        ops.rotary_tables(positions, inv_freq, torch.bfloat16)


def test_fractional_positions_keep_the_models_torch_ops():
    inv = 1.0 / (500000.0 ** (torch.arange(0, 64, 2) / 64))
    model = SimpleNamespace(_fused_ops=ops, inv_freq=inv, dtype=torch.bfloat16)
    cos, sin = RandomLlama._rotary(model, torch.tensor([[0.5, 3.25]]))
    want = torch.tensor([0.5, 3.25])[:, None] * torch.cat((inv, inv))
    assert torch.equal(cos[0], want.cos().to(torch.bfloat16)) and torch.equal(sin[0], want.sin().to(torch.bfloat16))


def _static(rows=8, cols=32, i64=torch.int64, i32=torch.int32):
    return [_gpu(rows, 1, dtype=i64), _gpu(rows, 1, dtype=i64), _gpu(1, rows, dtype=i64), _gpu(rows, cols, dtype=i64),
            _gpu(rows, dtype=i32)]


@pytest.mark.parametrize("n,cols,width,change", [
    (4, 5, 16, {}),  # padded past the buffers' rows
    (4, 5, 2, {}),
    (9, 5, 9, {}),
    (4, 33, 4, {}),  # wider than the table
    (4, 5, 8, {0: _gpu(4, 1, dtype=torch.int64)}),
    (4, 5, 8, {2: _gpu(1, 8, dtype=torch.int32)}),
    (4, 5, 8, {4: _gpu(8, dtype=torch.int64)}),
    (4, 5, 8, {3: _gpu(8, 32, dtype=torch.int32)}),
    (4, 5, 8, {3: _gpu(8, 64, dtype=torch.int64)[:, ::2]}),
    (4, 40, 8, {3: _gpu(8, 64, dtype=torch.int64)[:, :32]}),  # past the view, inside its rows
    (4, 0, 8, {3: _gpu(8, 0, dtype=torch.int64)}),
    (4, 5, 8, {1: _gpu(16, 1, dtype=torch.int64)[::2]}),
    (4, 5, 8, {1: torch.zeros(8, 1, dtype=torch.int64)}),
])
def test_a_step_that_does_not_fit_its_buffers_is_refused(n, cols, width, change):
    static = _static()
    for at, t in change.items():
        static[at] = t
    inputs = tuple(torch.zeros(*s, dtype=torch.int64) for s in ((n, 1), (n, 1), (1, n), (n, cols), (n,)))
    with pytest.raises(ValueError):
        ops.stage_decode(inputs, tuple(static), width, 0)


@pytest.mark.parametrize("n,cols", [(5, 3), (2, 17)])
def test_a_step_larger_than_the_captured_buffers_is_refused(n, cols):
    graphs = DecodeGraphs(SimpleNamespace(device=torch.device("cpu")), None, max_num_seqs=4, max_model_len=16, pad_slot=0)
    with pytest.raises(ValueError, match="does not fit the captured"):
        graphs.run(None, None, None, torch.zeros(n, cols, dtype=torch.int64), None)


@pytest.mark.parametrize("rows,n,k,served", [
    (128, 32768, 2048, True), (65, 24576, 1024, True),  # one round of 128-row tiles
    (65, 32776, 2048, False), (128, 40960, 1024, False), (128, 65408, 3584, False), (65, 65536, 3584, True),
    (96, 40960, 4096, False), (96, 49152, 4096, True), (128, 128256, 4096, True), (128, 128256, 2048, True),
    (33, 40960, 1024, False), (64, 49024, 3584, False), (64, 49152, 1024, True), (32, 40960, 1024, True),
    (128, 33000, 256, True), (128, 33024, 512, False),
])
def test_wide_weights_of_uneven_rounds_are_torchs(monkeypatch, rows, n, k, served):
    """256 CUs take 128-row tiles round by round; a nearly empty last round is left to torch's GEMM."""
    monkeypatch.undo()  # the rule itself
    assert (ops._splits(rows, n, k) > 0) == served
