"""The tiled GEMM's cost model, restated from the constants in csrc/tiled.hip: the token counts that
tests/test_gpu_short_tiles.py runs take the tiles it means, on the MI355X's 256 CUs, and the full-height
tiles serve the call it compares them with."""

from __future__ import annotations

import re
from pathlib import Path

import pytest

from test_gpu_short_tiles import CASES, DEPTHS, FULL

SOURCE = (Path(__file__).resolve().parent.parent / "llm-serving-engine_amd" / "csrc"
          / "tiled.hip").read_text()
CUS = 256


def _numbers(name: str) -> list[float]:
    body = re.search(rf"{name}\[kTileCands\] = \{{(.*?)\}};", SOURCE, re.S)[1]
    return [float(v) for v in re.findall(r"[\d.]+", body)]


def _constant(name: str) -> float:
    return float(re.search(rf"\b{name} = ([\d.]+)", SOURCE)[1])


_flat = [int(v) for v in _numbers("kTileCand")]
TILES = list(zip(_flat[::2], _flat[1::2]))
EFF = {"int8": _numbers("kTileEff16"), "w8a8": _numbers("kTileEff8")}


def _up(a: int, b: int) -> int:
    return -(-a // b)


def _cost(mode: str, glu: bool, m: int, n: int, k: int, i: int) -> float | None:
    (bm, bn), i8 = TILES[i], mode == "w8a8"
    if (bn == 192 and (i8 or glu)) or (bm == 96 and (i8 or m > 96)) or (bm == 112 and (i8 or not glu)):
        return None
    eff = EFF[mode][i]
    if i8 and bm == 192 and k < _constant("kShortKGlu" if glu else "kShortK"):
        eff = _constant("kTileEff8Short192")
    return _up(_up(m, bm) * _up(n, bn), CUS) * bm * bn / eff


def tile(mode: str, glu: bool, m: int, n: int, k: int) -> tuple[int, int]:
    """tiled_shape: the cheapest candidate, the earlier one within 0.1 %."""
    best, best_cost = None, float("inf")
    for i in range(len(TILES)):
        cost = _cost(mode, glu, m, n, k, i)
        if cost is not None and cost < best_cost * 0.999:
            best, best_cost = TILES[i], cost
    return best


@pytest.mark.parametrize("mode,glu,n,ms,rows", CASES)
@pytest.mark.parametrize("k", DEPTHS)
def test_short_tiles_are_taken(mode, glu, n, ms, rows, k):
    for m in ms:
        assert tile(mode, glu, m, n, k)[0] == rows, f"{m} tokens"
    assert tile(mode, glu, FULL, n, k)[0] in (64, 128, 256)


@pytest.mark.parametrize("glu,n,m,short,deep", [(True, 16384, 1152, 2048, 4096),
                                                (False, 5846, 3136, 2304, 3072)])
def test_few_k_steps_keep_the_small_tiles(glu, n, m, short, deep):
    """W8A8, where five rounds of 128 x 128 blocks meet two of 192 x 256: by the depth."""
    assert tile("w8a8", glu, m, n, short) == (128, 128)
    assert tile("w8a8", glu, m, n, deep) == (192, 256)
