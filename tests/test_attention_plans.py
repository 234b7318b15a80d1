"""How streaming decode attention cuts its keys (attn_stream_plan, host code): the change from four waves with ranges of 128 keys to eight with
256 is one line that a cache crosses once as it grows, not a band around some length."""
import ctypes as C
import importlib

import pytest

mynn = importlib.import_module("my-nn-engine_amd")


def plan(sequences, kv_heads, keys):
    """(keys of a range, ranges)"""
    rows, ranges = C.c_int(), C.c_int()
    mynn.lib()._ZN4mynn16attn_stream_planEiiiPiS0_(sequences, kv_heads, keys, C.byref(rows), C.byref(ranges))
    return rows.value, ranges.value


@pytest.mark.parametrize("pairs", [1, 2, 3, 4, 6, 8, 10, 12, 16, 20, 24, 31, 32, 48, 64, 100, 128, 255, 256, 300])
def test_longer_caches_do_not_go_back_to_short_ranges(pairs):
    """(two ranges of 128 keys are one of 256, which leaves nothing to merge: the one exception, below 257 keys)"""
    seen = 0
    for keys in range(257, 9000):
        rows, ranges = plan(pairs, 1, keys)
        assert rows % 128 == 0 and rows * ranges >= keys > rows * (ranges - 1)
        assert rows >= seen or rows >= 256, (keys, rows, seen)
        seen = max(seen, min(rows, 256))


def test_many_ranges_become_half_as_many():
    assert plan(4, 4, 1000) == (128, 8)
    for keys in (1200, 1500, 1800, 1920, 1921, 2048):  # (sixteen pairs: ten to sixteen ranges of 128 keys)
        assert plan(4, 4, keys) == (256, (keys + 255) // 256)
    assert plan(2, 4, 1500) == (128, 12)  # (eight pairs: they fill less than half of the device)
