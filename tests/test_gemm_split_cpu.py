"""The K split of the weight gradients' products, as the projection backward's
workspace shows it: 128 x 128 tiles take no fewer splits than the 64 x 64 tiles'
fill rule gives, so that no fp32 accumulator sums a longer chain for them."""

from __future__ import annotations

import ctypes

import pytest

from gru_qat_amd import _lib

CUS = 256


def _split(M, N, I):
    """Splits of dW [N, I] over M rows, from the workspace (dx unsplit: its rows are padded)."""
    off = _lib.GsQuant(*_lib._QOFF)
    a = _lib.GsProjBwdArgs(*([4096] * 7), 0, 0, M, N, I, I, N, I + 1, off, 0, 0, off)
    colsum = -(-(-(-M // 256) * N * 4) // 256) * 256
    parts = _lib.load().gs_input_proj_bwd_workspace_bytes(ctypes.byref(a)) - colsum
    assert parts >= 0
    return max(1, parts // (N * I * 4))


def _fill_split(M, N, I):
    tiles, smax = -(-N // 64) * -(-I // 64), max(1, min(16, -(-M // 256)))
    best, best_fill = 1, (-1, 1)
    for s in range(1, smax + 1):
        n = tiles * s
        if n < 2 * CUS and s < smax:
            continue
        fill = (n, CUS * -(-n // CUS))
        if fill[0] * best_fill[1] > best_fill[0] * fill[1]:
            best, best_fill = s, fill
    return best


@pytest.mark.parametrize("H,M", [(1924, 2052), (1929, 4282), (1001, 5300), (897, 16384), (512, 2048), (501, 1650)])
def test_split_never_lengthens_the_sums(H, M):
    assert _split(M, 3 * H, H) >= _fill_split(M, 3 * H, H)


def test_split_over_the_range():
    for H in range(16, 2049, 61):
        for M in (1, 256, 257, 1000, 2052, 4282, 5300, 16384, 32768):
            assert _split(M, 3 * H, H) >= _fill_split(M, 3 * H, H), (H, M)


def test_big_tiles_still_split_where_that_is_faster():
    assert _fill_split(32768, 3072, 1024) == 1 and _split(32768, 3072, 1024) == 4
