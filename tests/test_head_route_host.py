"""Which heads run on the tiled kernel: the rule alone, which needs no device."""
import pytest

from subspec_amd.model import tiled_head


@pytest.mark.parametrize("rows", [65, 96, 128])
def test_up_to_128_rows_the_length_of_a_row_decides(rows):
    """Rows of 8 KB from 96000 of them on; at longer ones neighbouring heads lie on both sides of the library GEMM."""
    for vocab in (96000, 99008, 128000, 130016, 140000, 147456, 152064, 158688, 201088, 262112):
        assert tiled_head(rows, vocab, 4096)
        assert not any(tiled_head(rows, vocab, hidden) for hidden in (2048, 3584, 4032, 4160, 4608, 5120, 8192))
    assert not tiled_head(rows, 90112, 4096) and not tiled_head(rows, 152064 + 16, 4096) and not tiled_head(rows, 262144, 4096)


def test_other_row_counts():
    assert not any(tiled_head(rows, 152064, 4096) for rows in (1, 64, 129, 192, 385))
    assert all(tiled_head(rows, 152064, 3584) for rows in (193, 289, 384)) and not tiled_head(321, 152064, 2048)
    assert tiled_head(193, 128256, 3072) and not tiled_head(193, 128256, 2048) and not tiled_head(193, 140000, 4096)
