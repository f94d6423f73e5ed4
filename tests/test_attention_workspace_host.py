"""Sizes of the attention workspace, from the library's host code alone."""
import pytest

from subspec_amd import _lib as L


def _bytes(batch, hq, hkv, rows, prefix, slots):
    return L.lib().subspec_tree_attention_workspace(batch, hq, hkv, rows, prefix, slots)


@pytest.mark.parametrize("hq,hkv", [(28, 4), (32, 8), (32, 32), (64, 8)])
@pytest.mark.parametrize("rows", [65, 128, 200, 289, 512])
def test_large_trees_hold_partials_only(hq, hkv, rows):
    """The fp32-sized partials of all rows in whole windows, at most 64 chunks of them; nothing that grows with the cache."""
    windows = (rows + 63) // 64
    for prefix in (100, 1300, 2048, 8192, 131072):
        chunks, rest = divmod(_bytes(1, hq, hkv, rows, prefix, rows), windows * hq * 64 * (128 * 4 + 8))
        assert rest in (0, 256) and chunks <= 64
    assert _bytes(1, hq, hkv, rows, 65536, rows) == _bytes(1, hq, hkv, rows, 262144, rows)


@pytest.mark.parametrize("batch,hq,hkv", [(1, 28, 4), (2, 28, 4), (8, 28, 4), (1, 14, 2), (2, 16, 8), (1, 32, 32), (5, 32, 8), (1, 64, 8)])
@pytest.mark.parametrize("rows", [1, 8, 16, 17, 40, 64, 289])
def test_a_workspace_serves_every_shorter_prefix(batch, hq, hkv, rows):
    """A captured call is laid out for the longest prefix it will see, and its workspace is held for calls of all shorter ones."""
    sizes = [_bytes(batch, hq, hkv, rows, prefix, rows) for prefix in range(0, 9000, 16)]
    assert sizes == sorted(sizes)
