"""Order of the causal attention's units, from the library's host code alone (the kernel evaluates the same function)."""
import ctypes

import pytest

from subspec_amd import _lib as L


def _order(hq, hkv, rows, prefix):
    n = L.lib().subspec_prefill_attention_order(hq, hkv, rows, prefix, None, 0)
    buf = (ctypes.c_int32 * (3 * n))()
    assert L.lib().subspec_prefill_attention_order(hq, hkv, rows, prefix, buf, n) == n
    return [tuple(buf[3 * i:3 * i + 3]) for i in range(n)]


@pytest.mark.parametrize("hq,hkv", [(28, 4), (16, 8), (32, 8), (2, 1), (64, 64)])
def test_every_chunk_once_and_long_ones_first(hq, hkv):
    falling = 0
    for rows in [*range(1, 200, 13), 63, 64, 65, 128, 256, 500, 1000, 1024, 1500, 1930, 2048, 4099, 8192]:
        for prefix in (0, 1, 63, 64, 65, 100, 511, 1000, 1792, 2048, 5000, 20001):
            order = _order(hq, hkv, rows, prefix)
            keys = order[0][2]
            windows = (rows + 63) // 64
            ends = [prefix + min(rows, 64 * (w + 1)) for w in range(windows)]
            needed = {(w, c) for w in range(windows) for c in range(-(-ends[w] // keys))}
            given = [(w, c) for w, c, _ in order if w >= 0]
            assert len(given) == len(set(given)), (rows, prefix)
            # more than needed: units whose first key lies behind the window's last one, which end at once
            assert needed <= set(given) and all(c * keys >= ends[w] for w, c in set(given) - needed), (rows, prefix)
            if windows * -(-ends[-1] // keys) * hkv * -(-(hq // hkv) // (8 if rows <= 32 else 4)) <= 256 or 2 * prefix > rows:
                assert given == [(w, c) for w in reversed(range(windows)) for c in range(-(-ends[-1] // keys))]
                continue
            falling += 1
            # the last window as if it had 64 rows: with fewer it may have a block less, but keeps its place
            blocks = [-(-min(keys, prefix + 64 * (w + 1) - c * keys) // 64) for w, c in given if (w, c) in needed]
            assert all(a >= b for a, b in zip(blocks, blocks[1:])), (rows, prefix, blocks)
            assert len(order) <= len(needed) + min(windows, keys // 64) + windows // (keys // 64) + 1
    assert falling >= 20


def test_sizes_that_no_prefill_has():
    order = L.lib().subspec_prefill_attention_order
    assert order(28, 5, 64, 0, None, 0) == -1 and order(28, 4, 0, 0, None, 0) == -1 and order(28, 4, 64, -1, None, 0) == -1
