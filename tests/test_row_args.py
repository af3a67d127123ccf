"""`ops._row_args`, the short cut of `ops._rows` for inputs whose memory already has the rows a kernel
takes, against it: the same address (or the same copied values), stride and count for every layout."""

from __future__ import annotations

import pytest
import torch


def _layouts():
    base = torch.arange(4096, dtype=torch.float32).to(torch.bfloat16)
    k = 32
    yield "1-D", base[:k]
    yield "rows", base[:4 * k].view(4, k)
    yield "one row", base[:k].view(1, k)
    yield "no rows", base[:0].view(0, k)
    yield "3-D", base[:6 * k].view(2, 3, k)
    yield "3-D with an empty dim", base[:0].view(2, 0, k)
    yield "columns of a wider matrix", base[:8 * 96].view(8, 96)[:, 32:64]
    yield "columns at an odd stride", base[:8 * 81].view(8, 81)[:, :32]
    yield "one row of a wider matrix", base[:96].view(1, 96)[:, 16:48]
    yield "misaligned", base[1:1 + 4 * k].view(4, k)
    yield "misaligned by 8 bytes", base[4:4 + 4 * k].view(4, k)
    yield "transposed", base[:4 * k].view(k, 4).t()
    yield "every second row", base[:8 * k].view(8, k)[::2]
    yield "permuted 3-D", base[:6 * k].view(3, 2, k).transpose(0, 1)
    yield "broadcast rows", base[:k].view(1, k).expand(5, k)


@pytest.mark.parametrize("name,x", list(_layouts()))
def test_agrees_with_rows(pkg, name, x):
    k = x.shape[-1]
    x2 = pkg.ops._rows(x, k)
    owner, at, ld, m = pkg.ops._row_args(x, k)
    assert m == x2.shape[0] and ld == (x2.stride(0) if m > 1 else k)
    assert at == owner.data_ptr()
    if x2.data_ptr() == x.data_ptr():
        assert at == x.data_ptr()
    else:
        assert at != x.data_ptr() and torch.equal(owner, x2)


def test_wrong_width_is_refused(pkg):
    with pytest.raises(RuntimeError, match="last dim"):
        pkg.ops._row_args(torch.zeros(4, 32, dtype=torch.bfloat16), 16)
