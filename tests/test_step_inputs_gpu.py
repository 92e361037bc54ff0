"""A step's inputs in one launch each: the rotary tables and a captured step's buffers, against the torch ops."""

from __future__ import annotations

import pytest
import torch

from liteinfer_amd.engine import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape,dim", [((1, 1), 64), ((1, 777), 128), ((256, 1), 128), ((3, 5), 2)])
def test_rotary_tables(shape, dim, dtype):
    g = torch.Generator(device="cuda").manual_seed(dim)
    positions = torch.randint(0, 131072, shape, generator=g, device="cuda")
    inv = 1.0 / (500000.0 ** (torch.arange(0, dim, 2, dtype=torch.float32, device="cuda") / dim))
    cos, sin = ops.rotary_tables(positions, inv, dtype)
    freqs = positions[..., None].float() * inv
    emb = torch.cat((freqs, freqs), -1)
    # The same fp32 argument; cosf / sinf within 2 ulp of each other's builds (2^-22 here), then
    # rounded: at most the neighbouring value, a spacing (eps) apart.
    tol = {torch.float32: 2.0 ** -22, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    for got, want in ((cos, emb.cos()), (sin, emb.sin())):
        assert got.shape == (*shape, dim) and got.dtype == dtype
        assert (got.double() - want.to(dtype).double()).abs().max() <= tol
        assert (got.double() - want.double()).abs().max() <= tol


@pytest.mark.parametrize("n,width,cols", [(1, 1, 1), (3, 4, 17), (24, 32, 900), (256, 256, 300)])
def test_stage_decode(n, width, cols):
    g = torch.Generator(device="cuda").manual_seed(n)
    rand = lambda *shape: torch.randint(5, 10 ** 6, shape, generator=g, device="cuda")  # noqa: E731
    inputs = (rand(n, 1), rand(n, 1), rand(1, n), rand(n, cols + 3)[:, 1:cols + 1], rand(n).to(torch.int32))
    rows, wide = 256, 1024
    static = (torch.full((rows, 1), -1, device="cuda"), torch.full((rows, 1), -1, device="cuda"),
              torch.full((1, rows), -1, device="cuda"), torch.full((rows, wide), -1, device="cuda"),
              torch.full((rows,), -1, dtype=torch.int32, device="cuda"))
    want = [t.clone() for t in static]
    for w, t in zip((want[0], want[1], want[2], want[4]), (inputs[0], inputs[1], inputs[2], inputs[4])):
        w.view(-1)[:n] = t.reshape(-1)
    want[3][:n, :cols] = inputs[3]
    for w, pad in ((want[0], 0), (want[1], 0), (want[2], 77), (want[4], 1)):
        w.view(-1)[n:width] = pad
    want[3][n:width, 0] = 77
    ops.stage_decode(inputs, static, width, 77)
    for got, w in zip(static, want):
        assert torch.equal(got, w)
    # Transposed and narrower inputs are taken as copies took them.
    ops.stage_decode((inputs[0], inputs[1].to(torch.int32), inputs[2], inputs[3].t().contiguous().t(), inputs[4]),
                     static, width, 77)
    for got, w in zip(static, want):
        assert torch.equal(got, w)
