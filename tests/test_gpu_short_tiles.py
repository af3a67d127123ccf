"""Token counts just past a block row run on tiles of 224, 192 or 112 token rows: every row has the
bits the full-height tiles give it (a 2048-token call of the same weight, whose rows sum K in the
same order), ragged last block rows, single and partial K steps included."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

FULL = 2048


@pytest.mark.parametrize("mode,glu,n,ms", [
    ("int8", True, 16384, (417, 448, 337)),   # 112 rows
    ("int8", True, 16384, (600, 576, 769)),   # 192 rows
    ("int8", False, 28672, (350, 384, 257)),  # 192 rows
    ("int8", False, 28672, (417, 448, 385)),  # 224 rows
    ("w8a8", True, 28672, (350, 384, 257)),   # 192 rows
    ("w8a8", True, 28672, (417, 448, 385)),   # 224 rows
    ("w8a8", False, 28672, (350, 417)),       # 192 and 224 rows
])
@pytest.mark.parametrize("k", [64, 144])
def test_rows_equal_the_full_tiles(pkg, dev, mode, glu, n, ms, k):
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
    if not glu and mode == "int8":
        ref = (x[:ms[0]].float() @ q.float().t()) * s
        err = (full[:ms[0]].float() - ref).abs().max()
        assert err <= 1e-2 * ref.abs().max()
