"""The decode step's projections (engine/ops.py: linear, linear_sums, gate_up_silu) against float64 products.

Sizes at the kernel's edges: one row, the row blocks of 16 / 32 / 64 / 128 / 256
and one past them, weight rows that fill no 128-row tile, one 128-k stage, and K cut
into many runs. `test_gate_up` also holds sizes that torch's GEMM serves;
`test_gate_up_through_every_kernel` names the kernels' own. Bound: the product of N(0, 1) x and 0.02 N(0, 1) w in fp32,
rounded once: half an ulp (at most 2^-8 relative in bf16, 2^-11 in fp16) plus fp32
summation error, well under 1e-4 here.
"""

from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

from liteinfer_amd.engine import ops

pytestmark = pytest.mark.gpu

ULP = {torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10}  # spacing of values, relative


def _inputs(rows, n, k, dtype):
    g = torch.Generator(device="cuda").manual_seed(rows * 7 + n + k)
    x = torch.randn(rows, k, generator=g, device="cuda").to(dtype)
    w = (torch.randn(n, k, generator=g, device="cuda") * 0.02).to(dtype)
    return x, w, x.double() @ w.double().t()


def _close(got, want, dtype):
    err = (got.double() - want).abs()
    assert (err <= 0.5 * ULP[dtype] * want.abs() + 1e-4).all(), err.max()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows", [1, 2, 15, 16, 17, 32, 33, 64, 65, 128, 129, 256])
@pytest.mark.parametrize("n,k", [(128, 128), (120, 256), (1000, 1152), (6144, 4096), (4088, 4096), (256, 14336), (33000, 256)])
def test_linear(rows, n, k, dtype):
    x, w, want = _inputs(rows, n, k, dtype)
    splits = ops._skinny(x, w)[1]
    if rows <= 64 or (n, k) == (6144, 4096) or (n, k, rows) in ((4088, 4096, 65), (4088, 4096, 129), (33000, 256, 128)):
        assert splits > 0  # (whole tiles, and runs in 128- and 64-row tiles, past 64 rows)
    _close(ops.linear(x, w), want, dtype)
    sums = ops.linear_sums(x, w)
    if isinstance(sums, ops.Partials):
        assert (sums.sums.double().sum(0) - want).abs().max() < 1e-4


@pytest.mark.parametrize("rows", [1, 16, 24, 64, 100, 200])
@pytest.mark.parametrize("ffn", [64, 1032, 14336])
def test_gate_up(rows, ffn):
    x, w, want = _inputs(rows, 2 * ffn, 512, torch.bfloat16)
    got = ops.gate_up_silu(x, w).double()
    gate, up = want.chunk(2, -1)
    # gate and up are rounded before the gate, its value before the product.
    tol = 4 * ULP[torch.bfloat16] * (F.silu(gate) * up).abs() + 2e-3 * (gate.abs() + up.abs()).clamp(min=1e-2)
    assert ((got - F.silu(gate) * up).abs() <= tol).all()
    # The same as the separate steps, the projection then the gate, up to the
    # order of the fp32 sums: gate, up, the gate's value and the product can
    # each round to the neighbour (a spacing apart, four in all), and where a
    # sum cancels its own error (512 terms of ~0.02: under 1e-5) shows whole.
    apart = ops.silu_mul(ops.linear(x, w)).double()
    assert ((got - apart).abs() <= 4 * ULP[torch.bfloat16] * apart.abs() + 1e-5 * (1 + up.abs() + gate.abs())).all()


@pytest.mark.parametrize("rows,splits", [(1, 2), (5, 8), (64, 13)])
def test_norm_adds_the_runs(rows, splits):
    g = torch.Generator(device="cuda").manual_seed(rows)
    sums = torch.randn(splits, rows, 1024, generator=g, device="cuda")
    h = torch.randn(rows, 1024, generator=g, device="cuda").to(torch.bfloat16)
    weight = torch.randn(1024, generator=g, device="cuda").to(torch.bfloat16)
    h2, delta = h.clone(), sums.double().sum(0)
    got = ops.add_rms_norm(h, weight, 1e-5, ops.Partials(sums, torch.Size((rows, 1024))))
    assert (h.double() - (h2.double() + delta)).abs().max() <= 2 ** -7 * (h2.double().abs() + delta.abs()).max()
    want = ops.add_rms_norm(h.clone(), weight, 1e-5)  # the norm of the row it left
    assert torch.equal(got, want)


def test_rows_it_does_not_serve_run_as_torch_products():
    x, w, want = _inputs(257, 256, 256, torch.bfloat16)
    assert ops._skinny(x, w)[1] == 0
    _close(ops.linear(x, w), want, torch.bfloat16)
    x, w, want = _inputs(4, 256, 192, torch.bfloat16)
    assert ops._skinny(x, w)[1] == 0
    odd = torch.zeros(4, 264, device="cuda", dtype=torch.bfloat16)[:, 4:260]
    assert ops._skinny(odd, torch.zeros(128, 256, device="cuda", dtype=torch.bfloat16))[1] == 0


@pytest.mark.parametrize("rows,ffn,k,splits", [
    (1, 1032, 512, 2), (24, 2048, 2048, 8), (64, 1032, 512, 2),  # skinny_gemm's gated sums
    (65, 2048, 4096, 4), (128, 2040, 4096, 4), (129, 2048, 4096, 4), (192, 2040, 4096, 4),  # 64-row tiles of batch_gemm
    (65, 2048, 14336, 8), (128, 2040, 14336, 8), (129, 2040, 14336, 8), (256, 2048, 14336, 8),  # 128-row tiles
    (65, 14336, 512, 1), (128, 12296, 512, 1),  # and whole ones, gated in the kernel
])
def test_gate_up_through_every_kernel(rows, ffn, k, splits):
    """Against float64, over the routes that the rule of the cut takes."""
    x, w, want = _inputs(rows, 2 * ffn, k, torch.bfloat16)
    assert ops._skinny(x, w)[1] == splits
    got = ops.gate_up_silu(x, w).double()
    gate, up = want.chunk(2, -1)
    out = F.silu(gate) * up
    # Half a spacing each for up, the gate's value and the product; the gate's
    # own moves silu by up to 1 + |gate| times as much. The fp32 sums: k terms
    # of ~0.02, under 1e-4.
    tol = (4 + gate.abs()) * 0.5 * ULP[torch.bfloat16] * out.abs() + 1e-4 * (1 + gate.abs() + up.abs())
    err = (got - out).abs()
    assert (err <= tol).all(), (err / tol).max()
