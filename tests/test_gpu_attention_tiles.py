"""The row-tiled paged attention of long entries on the GPU against the fp64 oracle, where it can go
wrong: the first entry length it takes, tiles of 128 rows and 64 keys one short and one over, groups
that do not divide a tile, block sizes a wave's 16 keys do and do not fit, short entries beside
long ones. The tolerance is test_gpu_attention's (bf16 probabilities and output)."""

from __future__ import annotations

import re
from pathlib import Path

import numpy as np
import pytest
import torch

from helpers import bf16_bits, to_bf16_tensor
from oracle import numerics as ora
from test_gpu_attention import _case, _check, _run

pytestmark = pytest.mark.gpu

HEADER = Path(__file__).resolve().parent.parent / "llm-serving-engine_amd" / "csrc" / "attention.h"
BOUND = {name: int(value) for name, value in
         re.findall(r"constexpr \w+ kAttnTile(\w+) = (\d+);", HEADER.read_text())}
WIDE = dict(h=160, h_kv=10)  # many heads, so that entries of 64 tokens are long


def _long(c, e):
    """Whether entry e of the case is the row-tiled kernel's, by the library's own bounds."""
    n, ctx, h, h_kv = int(c["ql"][e]), int(c["ctx"][e]), c["q"].shape[0], c["kp"].shape[2]
    start = "HeadsFew" if h_kv < 8 else "HeadsFar" if ctx > BOUND["Near"] else "Heads"
    return n * (h // h_kv) >= BOUND["Rows"] and (
        n * h >= BOUND["Always"]
        or (n * h >= BOUND[start] and n * h * (2 * ctx - n) >= 2 * BOUND["Pairs"]))


def _case_of(longs, *args, **kw):
    """A case of which exactly the entries `longs` are the row-tiled kernel's."""
    c = _case(*args, **kw)
    assert [e for e in range(len(c["ql"])) if _long(c, e)] == longs
    return c


@pytest.mark.parametrize("h,h_kv", [(40, 40), (30, 10), (32, 8), (50, 10), (96, 8), (128, 8)])
def test_first_length_and_tile_edges(pkg, dev, h, h_kv):
    """Entries on both sides of the first row-tiled length, and of the next row tile."""
    g = h // h_kv
    first = max(-(-BOUND["Always"] // h), -(-BOUND["Rows"] // g))
    tile = (first * g // 128 + 1) * 128
    lens = [first - 1, first, first + 1, tile // g, tile // g + 1]
    entries = [(n, off, n + off) for n, off in zip(lens, [0, 0, 3, 64, 129])]
    c = _case_of([1, 2, 3, 4], 100 + h, entries, h=h, h_kv=h_kv)
    _check(pkg, dev, c, f"H={h} H_KV={h_kv}")


def test_far_chunks_start_later(pkg, dev):
    """Entries on both sides of the bounds by context and by (row, key) pairs, whose tiles span many
    key steps."""
    entries = [(n, ctx - n, ctx) for n, ctx in [(128, 1040), (128, 1041), (127, 1100), (128, 4096),
                                                (128, 4097), (159, 4097), (160, 4097)]]
    _check(pkg, dev, _case_of([1, 3, 6], 150, entries, h=32, h_kv=8), "far chunks")
    entries = [(n, 900, n + 900) for n in (127, 128)]
    _check(pkg, dev, _case_of([1], 151, entries, h=64, h_kv=4), "few K/V heads")


@pytest.mark.parametrize("end", [63, 64, 65, 127, 128, 129, 191, 192, 193, 257])
def test_key_tile_edges(pkg, dev, end):
    """Contexts one short of and one over a key tile, a pair of tiles and the four in flight; the
    second entry's context ends before its own query rows do, so its rows see different ends."""
    c = _case_of([0, 1], 200 + end, [(end, 0, end), (end, 11, end)], h=176, h_kv=11)
    _check(pkg, dev, c, f"end={end}")


@pytest.mark.parametrize("block_size", [1, 7, 16, 24, 48, 64])
def test_block_sizes(pkg, dev, block_size):
    entries = [(150, 77, 227), (1, 300, 301), (64, 0, 64), (5, 100, 105)]
    c = _case_of([0, 2], 300 + block_size, entries, **WIDE, block_size=block_size)
    _check(pkg, dev, c, f"block {block_size}")


@pytest.mark.parametrize("log2_q", [2, 12, 40, -40])
def test_peaked_and_flat_scores(pkg, dev, log2_q):
    """Scores of which few keys, one key (from 2^12 on rounding the scaled maximum moves it by more than
    a probability's rounding, at 2^40 by more than fp32's range of exponents) and every key
    alike matter."""
    c = _case_of([0, 1], 450, [(150, 450, 600), (64, 0, 64)], **WIDE)
    c["q"] = ora.f32_to_bf16_bits(ora.bf16_bits_to_f32(c["q"]) * np.float32(2.0 ** log2_q))
    _check(pkg, dev, c, f"q x 2^{log2_q}")


def _errors(pkg, dev, c):
    """(relative error against fp64, the part of it that rounding the fp64 result to bf16 makes)."""
    o = ora.bf16_bits_to_f32(_run(pkg, dev, c)).astype(np.float64)
    golden, _ = ora.paged_attention_golden(c["q"], c["kp"], c["vp"], c["table"], c["ctx"], c["qo"],
                                           c["qs"], c["ql"], c["bs"])
    golden = np.asarray(golden, np.float64)
    rounded = ora.bf16_bits_to_f32(ora.f32_to_bf16_bits(golden.astype(np.float32)))
    rms = lambda a: float(np.sqrt((a ** 2).mean() / (golden ** 2).mean()))  # noqa: E731
    return rms(o - golden), rms(rounded - golden)


def test_the_largest_probabilities_are_exact(pkg, dev):
    """Few keys matter: each tile's largest probability is rounded to bf16 without error, so the
    relative error stays near that of the output's own rounding (0.00165). Over 1300 keys the other
    probabilities add 0.0003; with a reference that is not a whole number from the maximum they
    would all add 0.0014. The bound allows them 0.0007."""
    c = _case_of([0], 460, [(100, 1200, 1300)], **WIDE)
    c["q"] = ora.f32_to_bf16_bits(ora.bf16_bits_to_f32(c["q"]) * np.float32(3))
    error, rounding = _errors(pkg, dev, c)
    assert error <= np.hypot(rounding, 0.0007)


@pytest.mark.parametrize("tokens", [80, 417])
def test_rows_of_few_keys_keep_their_probabilities(pkg, dev, tokens):
    """A fresh prompt, whose first rows are the largest: beside the output's rounding (0.0016) its
    probabilities add 0.0003 at 80 tokens and 0.00075 at 417. Rounded to bf16 in those rows too they
    would add 0.0010 and 0.0011; the bounds lie between."""
    c = _case_of([0], 470 + tokens, [(tokens, 0, tokens)], h=128, h_kv=8)
    error, rounding = _errors(pkg, dev, c)
    assert error <= np.hypot(rounding, 0.0005 if tokens == 80 else 0.0009)


def test_rows_that_see_no_key(pkg, dev):
    """An entry without any context gives zeros."""
    c = _case_of([0, 1], 400, [(70, 0, 70), (80, 0, 80)], **WIDE)
    c["ctx"] = np.array([70, 0], np.int32)
    o = _run(pkg, dev, c)
    assert not (o[:, 70:] & 0x7FFF).any()
    assert (o[:, :70] & 0x7FFF).any()


def test_rows_do_not_depend_on_the_batch(pkg, dev):
    """A long entry's rows have the same bits alone, among decode rows and other prompts, with a
    larger max_q_len and a wider table; slots nobody owns hold NaN."""
    entries = [(1, 40, 41), (200, 100, 300), (90, 0, 90), (1, 700, 701), (65, 31, 96)]
    c = _case_of([1, 2, 4], 500, entries, **WIDE, spare_blocks=5)
    base = _check(pkg, dev, c, "batch")
    owned = np.zeros(c["kp"].shape[:2], bool)
    for e, ctx in enumerate(c["ctx"]):
        for n in range(ctx):
            owned[c["table"][e][n // c["bs"]], n % c["bs"]] = True
    kp, vp = c["kp"].copy(), c["vp"].copy()
    kp[~owned] = vp[~owned] = np.uint16(0x7FC0)
    np.testing.assert_array_equal(_run(pkg, dev, c, kp, vp), base, err_msg="NaN elsewhere")
    for e in (1, 2, 4):
        rows = slice(c["qs"][e], c["qs"][e] + c["ql"][e])
        pick = lambda a: a[e:e + 1]  # noqa: E731
        one = dict(c, q=c["q"][:, rows].copy(), table=np.pad(pick(c["table"]), ((0, 0), (0, 900))),
                   ctx=pick(c["ctx"]), qo=pick(c["qo"]), ql=pick(c["ql"]),
                   qs=np.zeros(1, np.int32), max_q_len=4000)
        np.testing.assert_array_equal(_run(pkg, dev, one), base[:, rows], err_msg=f"entry {e}")


def test_more_entries_than_one_launch_holds(pkg, dev):
    """Over 1024 entries, a few of them long."""
    longs = [e for e in range(1030) if e % 200 == 0 or e > 1026]
    entries = [(33, 0, 33) if e in longs else (1, 0, 1) for e in range(1030)]
    _check(pkg, dev, _case_of(longs, 600, entries, h=320, h_kv=20), "1030 entries")


@pytest.mark.parametrize("entries", [2, 32, 33, 63, 64, 65])
def test_entries_in_order_of_length(pkg, dev, entries):
    """Decode rows of different and equal contexts, with padding rows (q_len 0), on both sides of
    the entry counts whose workgroups are ordered by length and paired on a CU (from one more item
    than CUs to 64 entries)."""
    rng = np.random.default_rng(entries)
    ctx = rng.integers(1, 300, entries)
    ctx[0] = 300  # a table of more than 256 positions
    ctx[1::3] = 40
    c = _case(700 + entries, [(1, int(n) - 1, int(n)) for n in ctx], h=8, h_kv=8)
    base = _check(pkg, dev, c, f"{entries} entries")
    pad = dict(c, ql=c["ql"].copy(), ctx=c["ctx"].copy())
    pad["ql"][1::7] = pad["ctx"][1::7] = 0
    o = _run(pkg, dev, pad)
    keep = pad["ql"] > 0
    np.testing.assert_array_equal(o[:, keep], base[:, keep])


def _indexes(c, dev):
    return [torch.from_numpy(np.ascontiguousarray(c[k], np.int32)).to(dev)
            for k in ("table", "ctx", "qo", "qs", "ql")]


@pytest.mark.parametrize("block_size", [16, 24])
@pytest.mark.parametrize("pools", ["padded rows", "head-major blocks"])
def test_layouts(pkg, dev, block_size, pools):
    """q as columns of a stacked projection, token-major, with o in its order, and pools of other
    strides: the bits of the contiguous call, long and short entries."""
    entries = [(70, 30, 100), (1, 60, 61), (5, 0, 5), (64, 0, 64)]
    c = _case_of([0, 3], 800 + block_size, entries, **WIDE, block_size=block_size)
    want = _check(pkg, dev, c, "contiguous")
    h, tokens, d = c["q"].shape
    stacked = torch.zeros(tokens, (h + 20) * d, dtype=torch.bfloat16, device=dev)
    q = stacked[:, :h * d].view(tokens, h, d).transpose(0, 1)
    q.copy_(to_bf16_tensor(c["q"], dev))
    kv = []
    for name in ("kp", "vp"):
        pool = to_bf16_tensor(c[name], dev)
        blocks, slots, heads, _ = pool.shape
        if pools == "padded rows":
            view = torch.full((blocks, slots, heads, 2 * d), float("nan"), dtype=pool.dtype,
                              device=dev)[..., :d]
        else:
            view = torch.empty(blocks, heads, slots, d, dtype=pool.dtype, device=dev).transpose(1, 2)
        kv.append(view.copy_(pool))
    o = pkg.ops.paged_attention_forward(q, *kv, *_indexes(c, dev), c["bs"], c["max_q_len"])
    np.testing.assert_array_equal(bf16_bits(o), want)


def _with_scale(pkg, dev, c, scale):
    q, k, v = (to_bf16_tensor(c[n], dev) for n in ("q", "kp", "vp"))
    table, ctx, qo, qs, ql = _indexes(c, dev)
    o = torch.empty_like(q)
    lib, (h, _, d), h_kv = pkg.library(), q.shape, k.shape[2]
    shape = (len(ctx), h, h_kv, d)
    nbytes = lib.lse_paged_attention_workspace_bytes(*shape, c["max_q_len"], table.shape[1], c["bs"])
    ws = torch.empty(max(nbytes, 16), dtype=torch.uint8, device=dev)
    status = lib.lse_paged_attention(
        q.data_ptr(), q.stride(0), q.stride(1), k.data_ptr(), v.data_ptr(), *k.stride()[:3],
        table.data_ptr(), table.stride(0), ctx.data_ptr(), qo.data_ptr(), qs.data_ptr(),
        ql.data_ptr(), o.data_ptr(), o.stride(0), o.stride(1), *shape, c["bs"], table.shape[1],
        c["max_q_len"], scale, ws.data_ptr(), nbytes, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert status == 0
    return bf16_bits(o)


def test_negative_and_zero_scales(pkg, dev):
    """The C entry's softmax scale of either sign, and none: the bits of the negated and of zero queries
    under a positive one, long and short entries."""
    c = _case_of([0], 820, [(70, 30, 100), (5, 40, 45), (1, 99, 100)], **WIDE)
    np.testing.assert_array_equal(_with_scale(pkg, dev, c, -0.125),
                                  _with_scale(pkg, dev, dict(c, q=c["q"] ^ 0x8000), 0.125))
    np.testing.assert_array_equal(_with_scale(pkg, dev, c, 0.0),
                                  _with_scale(pkg, dev, dict(c, q=np.zeros_like(c["q"])), 0.125))


@pytest.mark.parametrize("key", [0, 20, 64, 130])
def test_infinite_scores(pkg, dev, key):
    """A score of -inf leaves its key out; one of +inf makes the rows that see it NaN, and no other."""
    c = _case_of([0, 1], 830, [(150, 0, 150), (64, 0, 64)], **WIDE)
    c["q"][:, :, 0] = 0x3F80  # 1.0
    clean = _run(pkg, dev, c)
    at = (c["table"][0][key // c["bs"]], key % c["bs"])
    c["kp"] = c["kp"].copy()
    c["kp"][at[0], at[1], :, 0] = 0xFF80  # -inf
    left_out = _run(pkg, dev, c)
    golden, covered = ora.paged_attention_golden(
        c["q"], np.where(c["kp"] == 0xFF80, np.uint16(0xFF7F), c["kp"]), c["vp"], c["table"],
        c["ctx"], c["qo"], c["qs"], c["ql"], c["bs"])
    if key == 0:  # its own row sees no other key
        assert not (left_out[:, 0] & 0x7FFF).any()
        covered = covered.copy()
        covered[0] = False
    vmax = float(np.abs(ora.bf16_bits_to_f32(c["vp"])).max())
    ok, msg = ora.attention_within_tolerance(left_out, golden, vmax, covered)
    assert ok, msg
    c["kp"][at[0], at[1], :, 0] = 0x7F80  # +inf
    o = ora.bf16_bits_to_f32(_run(pkg, dev, c))
    assert np.isnan(o[:, key:150]).all()
    np.testing.assert_array_equal(ora.f32_to_bf16_bits(o[:, :key]), clean[:, :key])
    np.testing.assert_array_equal(ora.f32_to_bf16_bits(o[:, 150:]), clean[:, 150:])


@pytest.mark.parametrize("bad", [0x7FC0, 0x7F80])
def test_how_far_a_non_finite_v_row_reaches(pkg, dev, bad):
    """NaN or infinity in a token's V: NaN or infinite for the rows that see it, no trace in the rows of
    earlier row tiles (8 tokens of 16 heads), other K/V heads and other entries."""
    c = _case_of([0, 1], 840, [(70, 0, 70), (64, 0, 64)], **WIDE)
    clean = _run(pkg, dev, c)
    token, head = 44, 3
    vp = c["vp"].copy()
    vp[c["table"][0][token // c["bs"]], token % c["bs"], head] = bad
    o = _run(pkg, dev, c, vp=vp)
    group = slice(16 * head, 16 * head + 16)
    assert not np.isfinite(ora.bf16_bits_to_f32(o[group, token:70])).any()
    same = np.ones(o.shape[:2], bool)
    same[group, token // 8 * 8:70] = False
    np.testing.assert_array_equal(o[same], clean[same])


@pytest.mark.parametrize("max_q_len", [9000, 40000, 100000])
def test_work_list_of_grouped_row_tiles(pkg, dev, max_q_len):
    """A max_q_len whose row tiles exceed the work list's levels (1024) puts several tiles into one: the
    same bits as with the exact one."""
    c = _case_of([0, 2, 3], 850, [(150, 77, 227), (1, 300, 301), (64, 0, 64), (333, 0, 333)], **WIDE)
    base = _check(pkg, dev, c, "exact max_q_len")
    np.testing.assert_array_equal(_run(pkg, dev, dict(c, max_q_len=max_q_len)), base)


def test_more_items_than_a_workgroup_lists_at_once(pkg, dev):
    """1024 entries of 136 items: over 512 for each of 256 workgroups, so that the lists are filled twice.
    Every entry has the bits it has in a call of 64."""
    h, h_kv, d, n, count, bs = 32, 8, 128, 520, 1024, 16
    gen = torch.Generator(device=dev).manual_seed(860)
    bf16 = lambda *shape: torch.randn(*shape, generator=gen, device=dev,  # noqa: E731
                                      dtype=torch.bfloat16)
    blocks = -(-n // bs)
    k, v, q = bf16(blocks, bs, h_kv, d), bf16(blocks, bs, h_kv, d), bf16(count * n, h, d)
    full = lambda m, value: torch.full((m,), value, dtype=torch.int32, device=dev)  # noqa: E731

    def run(rows, m):
        table = torch.arange(blocks, dtype=torch.int32, device=dev).repeat(m, 1)
        start = torch.arange(0, m * n, n, dtype=torch.int32, device=dev)
        return pkg.ops.paged_attention_forward(rows.transpose(0, 1), k, v, table, full(m, n),
                                               full(m, 0), start, full(m, n), bs, n).transpose(0, 1)

    o = run(q, count)
    for e in range(0, count, 64):
        rows = slice(e * n, (e + 64) * n)
        assert torch.equal(o[rows], run(q[rows], 64)), f"entries from {e}"
