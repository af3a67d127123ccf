"""Token counts just past a block row run on tiles of 224, 192 or 112 token rows: every row has the
bits the full-height tiles give it (a 2048-token call of the same weight, whose rows sum K in the
same order), ragged last block rows and partial K steps included, with fewer K steps than stage
slots, and with many more, whose slots are refilled while other waves still read theirs; and the rows
agree with a product in fp64. tests/test_tile_model.py checks which tile each count takes."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

FULL = 2048
CASES = [  # mode, gate/up, N (of both halves in gate/up: I), token counts, their tile's rows
    ("int8", True, 16384, (417, 448, 337), 112),
    ("int8", True, 16384, (600, 576, 513), 192),
    ("int8", True, 16384, (769, 896), 224),
    ("int8", False, 28672, (350, 384, 257), 192),
    ("int8", False, 28672, (417, 448, 385), 224),
    ("w8a8", True, 28672, (350, 384, 257), 192),
    ("w8a8", True, 28672, (417, 448, 385), 224),
    ("w8a8", False, 28672, (350,), 192),
    ("w8a8", False, 28672, (417,), 224),
]
DEPTHS = [64, 144, 1040, 4112]  # 1, 3, 17 and 65 steps of 64


def _golden(ops, mode, glu, x, q, s):
    """fp64: s (x q), in W8A8 with the library's own quantized x (tests/test_gpu_quant.py); gate/up
    silu(g) u."""
    if mode == "w8a8":
        xq, sx = ops.quantize_act_per_token(x)
        x = xq.double() * sx.double()[:, None]
    x = x.double()
    y = (x @ q.double().t().contiguous()) * s.double()
    if glu:
        g, u = y.chunk(2, 1)
        y = g / (1 + torch.exp(-g)) * u
    return y


@pytest.mark.parametrize("mode,glu,n,ms,rows", CASES)
@pytest.mark.parametrize("k", DEPTHS)
def test_rows_equal_the_full_tiles(pkg, dev, mode, glu, n, ms, rows, k):
    gen = torch.Generator(device=dev).manual_seed(n + k)
    x = torch.randn(FULL, k, generator=gen, device=dev).to(torch.bfloat16)
    q = torch.randint(-127, 128, (n, k), generator=gen, device=dev, dtype=torch.int8)
    s = torch.rand(n, generator=gen, device=dev) * 1e-2
    ops = pkg.ops
    if glu:
        qp = ops.pack_glu(q)
        call = {"int8": ops.w8a16_glu, "w8a8": ops.w8a8_glu}[mode]
    else:
        qp = ops.pack_weight(q)
        call = {"int8": ops.w8a16_linear, "w8a8": ops.w8a8_linear}[mode]
    full = call(x, qp, s)
    for m in ms:
        assert torch.equal(call(x[:m].contiguous(), qp, s), full[:m]), f"{m} tokens"
    # The output's rounding to bf16 (2^-9 of a value) and fp32 sums of k products (k 2^-24 of the sum
    # of their magnitudes, about sqrt(k) of the result's size), the latter through the product of
    # gate/up's two halves as well.
    want = _golden(ops, mode, glu, x[:ms[0]], q, s)
    got = call(x[:ms[0]].contiguous(), qp, s).double()
    size = want.square().mean().sqrt()
    assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + 1e-3 * size).all()
