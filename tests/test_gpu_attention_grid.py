"""Paged attention of short entries on the GPU: every order of the grid takes each (entry, K/V head, query
tile, key chunk) item exactly once. Entries of one and of several query tiles, padding entries
(q_len 0) among them, entry counts on both sides of the bounds between the orders, and the same
rows' bits in each of them. The tolerance is test_gpu_attention's."""

from __future__ import annotations

import numpy as np
import pytest

from test_gpu_attention import _case, _check, _run

pytestmark = pytest.mark.gpu


def _entries(count, several, ctx):
    """`count` entries, every `several`-th of 3 to 20 query rows, the others of one."""
    rng = np.random.default_rng(count * several + ctx)
    out = []
    for e in range(count):
        rows = int(rng.integers(3, 21)) if e % several == 0 else 1
        end = int(rng.integers(rows, ctx + rows))
        out.append((rows, end - rows, end))
    return out


@pytest.mark.parametrize("count,several,ctx", [
    (2, 2, 90), (16, 5, 90), (17, 1, 40), (17, 17, 90), (40, 3, 60), (63, 9, 90), (64, 64, 400),
    (65, 5, 60), (130, 4, 40),  # unsplit: the first tiles first, or compact from 17 to 64 entries
    (1, 1, 2500), (3, 2, 2500), (9, 4, 2500),  # split over chunks
])
@pytest.mark.parametrize("h,h_kv", [(16, 8), (6, 2)])
def test_every_item_is_taken(pkg, dev, count, several, ctx, h, h_kv):
    c = _case(800 + count + several, _entries(count, several, ctx), h=h, h_kv=h_kv)
    base = _check(pkg, dev, c, f"{count} entries, every {several}th of several tiles")
    pad = dict(c, ql=c["ql"].copy(), ctx=c["ctx"].copy())
    pad["ql"][1::6] = pad["ctx"][1::6] = 0
    keep = np.repeat(pad["ql"] > 0, c["ql"])
    o = _run(pkg, dev, pad)
    np.testing.assert_array_equal(o[:, keep], base[:, keep], err_msg="with padding entries")


def test_rows_have_the_same_bits_in_every_order(pkg, dev):
    """Three entries alone (split over their chunks), among 20 and among 70 entries (unsplit)."""
    few = [(20, 1500, 1520), (1, 2000, 2001), (7, 30, 37)]
    others = [(1, 5, 6)] * 67
    c = _case(900, few + others, h=16, h_kv=8)
    base = _check(pkg, dev, c, "70 entries")
    for n in (3, 20):
        rows = int(c["ql"][:n].sum())
        part = dict(c, q=c["q"][:, :rows].copy(),
                    **{k: c[k][:n].copy() for k in ("table", "ctx", "qo", "qs", "ql")})
        np.testing.assert_array_equal(_run(pkg, dev, part), base[:, :rows], err_msg=f"{n} entries")
