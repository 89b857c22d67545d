"""The backward's workspace without a GPU: what the pools' gradient adds to it."""

from __future__ import annotations

import ctypes

import pytest

from dsv4_planb_amd import _lib
from tests.test_capi import _good

BOUND = 2 << 30  # bytes of spilled P and dS and of inverse lists per run of tokens


def _size(p, kv_grad):
    n = ctypes.c_size_t()
    assert _lib.load().sas_backward_workspace_size_for(ctypes.byref(p), kv_grad, ctypes.byref(n)) == 0
    return n.value


# whole groups of 64 tokens would pass the bound (250 and 700 tokens); fit it (8192); one
# short run (96); fewer than 8 tokens per sequence: nothing is spilled
@pytest.mark.parametrize("T,B,H,topk", [(250, 1, 128, 40000), (700, 2, 100, 25000), (8192, 4, 128, 512),
                                        (96, 1, 16, 64), (15, 2, 64, 512)])
def test_the_spill_keeps_to_its_bound(T, B, H, topk):
    p = _good(total_tokens=T, batch=B, num_heads_q=H, topk=topk, cmp_table_len=64, cmp_block_size=128,
              cmp_block_stride=128 * 576)
    extra = _size(p, 1) - _size(p, 0)
    total = ctypes.c_size_t()
    assert _lib.load().sas_backward_workspace_size(ctypes.byref(p), ctypes.byref(total)) == 0
    assert total.value == _size(p, 1)
    if T < 8 * B:
        assert extra == 0
        return
    cmp_rows = 64 * 128 if 64 * 128 <= 6 * topk else 0
    rows = topk if cmp_rows else 0
    per_token = (128 + rows + 31) // 32 * 32 * ((H + 31) // 32 * 128) + 4 * cmp_rows
    # beside them: a flag per token, the items (at most one per 8 tokens and sequence and per
    # tile) and each region's alignment
    tiles = (127 + 64) // 128 + 2 + (cmp_rows + 127) // 128
    beside = 4 * (T + 1) + 16 * ((T // 8 + B + 1) * tiles + 1) + 4 * 256
    assert extra <= min(BOUND, T * per_token) + per_token // 100 + 1024 + beside
    assert extra >= min(BOUND // 2, T * per_token) - per_token


# tables of 6 K compressed rows (the most that tiles take): inverse lists of every token would
# be 3 to 9 GiB
@pytest.mark.parametrize("T,B,H", [(65536, 1, 128), (131072, 4, 128), (200000, 1, 16)])
def test_long_calls_keep_to_the_bound(T, B, H):
    p = _good(total_tokens=T, batch=B, num_heads_q=H, topk=2048, cmp_table_len=96, cmp_block_size=128,
              cmp_block_stride=128 * 576)
    extra = _size(p, 1) - _size(p, 0)
    assert extra > BOUND // 2  # (tiles for the compressed rows)
    # the flags, and at most an item per 8 tokens of a run and per tile (12288 / 128 + 3)
    run = BOUND // (2176 * ((H + 31) // 32 * 128) + 4 * 12288)
    assert extra <= BOUND + 4 * (T + 1) + 16 * ((run // 8 + B + 1) * 99 + 1) + 8 * 256
