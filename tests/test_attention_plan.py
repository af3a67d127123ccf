"""When paged attention splits its rows over key chunks, from the workspace the split needs (without a GPU
the library plans for the MI355X's 256 CUs)."""

from __future__ import annotations

import pytest


def _workspace(pkg, entries, h, h_kv, max_q_len, positions, block_size=16):
    return pkg.library().lse_paged_attention_workspace_bytes(
        entries, h, h_kv, 128, max_q_len, positions // block_size, block_size)


@pytest.mark.parametrize("h,h_kv,max_q_len", [(32, 8, 2048), (32, 8, 512), (24, 8, 1024),
                                              (8, 2, 1024), (4, 1, 2048)])
@pytest.mark.parametrize("positions", [4096, 65536])
def test_a_prompt_chunk_is_not_split(pkg, h, h_kv, max_q_len, positions):
    """One entry whose query tiles fill the CUs twice over needs no workspace, however wide its table."""
    assert _workspace(pkg, 1, h, h_kv, max_q_len, positions) == 0


def test_few_rows_over_a_long_context_are_split(pkg):
    chunks, rows = 4, 32
    assert _workspace(pkg, 1, 32, 8, 1, 4096) == chunks * rows * (128 + 2) * 4
    assert _workspace(pkg, 1, 32, 8, 1, 1024) == 0  # one chunk
    assert _workspace(pkg, 64, 32, 8, 1, 4096) == 0  # 512 items
